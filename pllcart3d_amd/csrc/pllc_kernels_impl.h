// pllc_kernels_impl.h -- the HIP kernels of one pllcart3d RK3-CN substage
// and their launch layer, templated on the field type T.
//
// Every kernel restates one reference routine (cited per kernel) with the
// same operand order.  This file is compiled twice: pllc_kernels_f64.hip
// instantiates T = double with -ffp-contract=off (the reference arithmetic
// operation by operation), pllc_kernels_f32.hip instantiates T = float with
// contraction and fast division (the mixed path).  PLLC_F64_TU selects the
// instantiation and the FP64-only helpers of the Tds / fftw entry points.
#pragma once
#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <utility>

#include "pllc_dev.h"
#include "pllc_grid.h"
#include "pllc_host.h"
#include "pllc_kernels.h"

namespace pllc {

// The member of a batched launch (Bt) whose block has index idx along the
// grid dimension of size dim that carries the members (nm equal ranges),
// and the block's index within its member's range.
__device__ __forceinline__ int bt_member(const Bt& bt, unsigned idx, unsigned dim, int& local)
{
    const int per = (int)(dim / (unsigned)bt.nm);
    const int m = (int)idx / per;
    local = (int)idx - m * per;
    return m;
}
// member m's copy of a field pointer (null stays null)
template <typename T>
__device__ __forceinline__ T* bt_f(const Bt& bt, T* p, int m)
{
    return p ? p + (long)m * bt.fs : p;
}
// member m's physics: the launch's own argument, or with B (a batched
// launch; a compile-time choice, so that the single form keeps its
// registers) the batch's table
template <bool B>
__device__ __forceinline__ const Phys& bt_phys(const Bt& bt, const Phys& own, int m);
template <>
__device__ __forceinline__ const Phys& bt_phys<false>(const Bt&, const Phys& own, int)
{
    return own;
}
template <>
__device__ __forceinline__ const Phys& bt_phys<true>(const Bt& bt, const Phys&, int m)
{
    return bt.ph[m];
}
template <typename T>
__device__ __forceinline__ Visc4<T> bt_mu(const Bt& bt, const Visc4<T>& mu, int m)
{
    return {bt_f(bt, mu.cell, m), bt_f(bt, mu.xy, m), bt_f(bt, mu.xz, m), bt_f(bt, mu.yz, m)};
}

// ------------------------------------------------------------ stale D2

// The ENO boundary rule of Hc/Hu/Hv/Hw_op reads D2 one index outside the
// range its pass just wrote and sees what an earlier pass of the same call
// left in the shared scratch array (pllcart3d.c:1546, 1568, 1596, 1626).
// For every operator f (c,u,v,w) and pass (y,z) this kernel computes the
// two values such reads return: [f*4 + 0] y-pass at js-1, [+1] y-pass at
// je+1, [+2] z-pass at ks-1, [+3] z-pass at ke+1.  The x pass runs first on
// a zeroed scratch, so its outside reads are 0.
template <typename T>
__device__ __forceinline__ T stale_value(const Dims& d, const T* __restrict__ q0, const T* __restrict__ q1,
                                         const T* __restrict__ q2, const T* __restrict__ q3, int t)
{
    const int f = t >> 2, w = t & 3;
    const T* q = f == 0 ? q0 : f == 1 ? q1 : f == 2 ? q2 : q3;
    const Rng R = field_rng(d, f);
    const T hx = T(d.dx), hy = T(d.dy);
    // D2 of the x pass's last line (j = je, k = ke) and of the y pass's last
    // line (i = ie, k = ke), at index m
    const T* px = q + IX(d, 0, R.je, R.ke);
    const T* py = q + IX(d, R.ie, 0, R.ke);
    T v = T(0.0);
    if (w < 2) {
        const int m = w == 0 ? R.js - 1 : R.je + 1;
        if (m >= R.is && m <= R.ie)
            v = divh<T>(dd1(px, d.sx, m, hx, d.rdx) - dd1(px, d.sx, m - 1, hx, d.rdx), T(2.0) * hx, 0.5 * d.rdx);
    } else {
        const int m = w == 2 ? R.ks - 1 : R.ke + 1;
        if (m >= R.js && m <= R.je)
            v = divh<T>(dd1(py, d.sy, m, hy, d.rdy) - dd1(py, d.sy, m - 1, hy, d.rdy), T(2.0) * hy, 0.5 * d.rdy);
        else if (m >= R.is && m <= R.ie)
            v = divh<T>(dd1(px, d.sx, m, hx, d.rdx) - dd1(px, d.sx, m - 1, hx, d.rdx), T(2.0) * hx, 0.5 * d.rdx);
    }
    return v;
}

template <typename T>
__global__ void k_stale(Dims d, const T* __restrict__ q0, const T* __restrict__ q1, const T* __restrict__ q2,
                        const T* __restrict__ q3, T* __restrict__ stale)
{
    const int t = threadIdx.x;
    if (t < 16) stale[t] = stale_value<T>(d, q0, q1, q2, q3, t);
}

// ------------------------------------------------- explicit terms + source

// XCD-aware tile order of the cell grids (blocks of 128 k x 2 j or 64 k x
// 4 j, grid (k tiles, j tiles, planes)).  Workgroups go to the 8 XCDs round-robin by
// linear id and each XCD has its own L2.  In dispatch order a plane's
// consecutive j tiles land on different XCDs, so every XCD fetches the
// y-stencil halo rows of its tiles itself.  This hands XCD x the x-th eighth
// of each plane's tiles in (k, j) order instead, a band of consecutive j
// rows, whose halo rows its L2 shares; planes keep their dispatch order, so
// the x-stencil planes stay in the same L2 as before.  A bijection of the
// plane's tiles (the identity when their count is not a multiple of 8).
__device__ __forceinline__ int2 xcd_tile()
{
    const int gx = gridDim.x, nt = gx * gridDim.y;
    int r = blockIdx.x + gx * blockIdx.y;
    if ((nt & 7) == 0) r = (r & 7) * (nt >> 3) + (r >> 3);
    return make_int2(r % gx, r / gx);
}

// The field value uo values after p at the lane's byte offset v: p + uo is
// uniform over the block and stays in scalar registers, v is the one vector
// register all loads of a thread share.  (A plane of 2^32 bytes would need
// fields larger than the device's memory.)
template <typename T>
__device__ __forceinline__ const T& lane_at(const T* __restrict__ p, long uo, unsigned v)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p + uo) + v);
}
template <typename T>
__device__ __forceinline__ T& lane_at(T* __restrict__ p, long uo, unsigned v)
{
    return *reinterpret_cast<T*>(reinterpret_cast<char*>(p + uo) + v);
}

// The lane offset anew in a loop's block: its widening to 64 bits then stays
// beside the loads and stores, which take the 32-bit register as it is
// (widened once before the loop it costs an addition per access).
__device__ __forceinline__ void per_block(unsigned& v, long& o) { asm("" : "+v"(v), "+s"(o)); }

// Consecutive points in k that a thread of the explicit kernels takes: an
// 8-byte load of a wave occupies the L1's address unit for 17 cycles, a
// 16-byte load (any 8-byte alignment) for the same 17, a 4-byte load for 5
// (measured, all L1 hits), so FP64 threads take two points and FP32 threads
// one.
template <typename T> struct KP { static constexpr int value = sizeof(T) == 8 ? 2 : 1; };

// n consecutive values at the lane's address, in 16-byte pieces in FP64
typedef double dpair __attribute__((ext_vector_type(2), aligned(8)));
template <int n>
__device__ __forceinline__ void lane_run(const double* __restrict__ p, long uo, unsigned v, double (&a)[n])
{
#pragma unroll
    for (int t = 0; t + 1 < n; t += 2) {
        const dpair x = *reinterpret_cast<const dpair*>(&lane_at(p, uo + t, v));
        a[t] = x.x;
        a[t + 1] = x.y;
    }
    if (n & 1) a[n - 1] = lane_at(p, uo + n - 1, v);
}
template <int n>
__device__ __forceinline__ void lane_run(const float* __restrict__ p, long uo, unsigned v, float (&a)[n])
{
#pragma unroll
    for (int t = 0; t < n; t++) a[t] = lane_at(p, uo + t, v);
}
// the lane's values of k .. k + KP - 1 that lie in ks .. ke to the field
__device__ __forceinline__ void lane_put(double* __restrict__ p, long uo, unsigned v, const double (&a)[2], int k,
                                         int ks, int ke)
{
    if (k >= ks && k < ke) {
        dpair x;
        x.x = a[0];
        x.y = a[1];
        *reinterpret_cast<dpair*>(&lane_at(p, uo, v)) = x;
    } else {
        if (k >= ks && k <= ke) lane_at(p, uo, v) = a[0];
        if (k + 1 >= ks && k + 1 <= ke) lane_at(p, uo + 1, v) = a[1];
    }
}
__device__ __forceinline__ void lane_put(float* __restrict__ p, long uo, unsigned v, const float (&a)[1], int, int, int)
{
    lane_at(p, uo, v) = a[0];
}

// the seven values around each of a thread's points: along x from the planes
// it carries, along y from the rows around it, along z from its own run of
// KP + 6 values
template <typename T>
struct Cross {
    static constexpr int K = KP<T>::value;
    T x[7][K], y[7][K], lo[3], hi[3];
    // the planes i - 3 .. i + 2 as if i - 1 had been done
    __device__ __forceinline__ void start(const T* __restrict__ q, long o, unsigned v, long sx)
    {
#pragma unroll
        for (int m = 1; m < 7; m++) lane_run(q, o + (long)(m - 4) * sx, v, x[m]);
    }
    // to plane i at o
    __device__ __forceinline__ void next(const T* __restrict__ q, long o, unsigned v, long sx, long sy)
    {
#pragma unroll
        for (int m = 0; m < 6; m++)
#pragma unroll
            for (int p = 0; p < K; p++) x[m][p] = x[m + 1][p];
        lane_run(q, o + 3 * sx, v, x[6]);
#pragma unroll
        for (int m = 0; m < 7; m++)
            if (m != 3) lane_run(q, o + (long)(m - 3) * sy, v, y[m]);
        lane_run(q, o - 3, v, lo);
        lane_run(q, o + K, v, hi);
    }
    // the stencils of point p
    __device__ __forceinline__ void at(int p, T (&sx7)[7], T (&sy7)[7], T (&sz7)[7]) const
    {
#pragma unroll
        for (int m = 0; m < 7; m++) {
            sx7[m] = x[m][p];
            sy7[m] = m == 3 ? x[3][p] : y[m][p];
            const int t = p + m;   // of the run k - 3 .. k + K + 2
            sz7[m] = t < 3 ? lo[t] : t < 3 + K ? x[3][t - 3] : hi[t - 3 - K];
        }
    }
};

// concentration's explicit part at the points i .. ie of one j and KP
// consecutive k: Hc_op (1539-1644) and the source loop (573-590).  From plane
// to plane the x stencil and the upper face's u stay in registers.
template <typename T, bool FAST>
__device__ __forceinline__ void rhs_conc_line(const Dims& d, const Phys& ph, const Rng& R, int i, int ie, int j, int k0,
                                              long mo, const T* __restrict__ cold, const T* __restrict__ un,
                                              const T* __restrict__ vn, const T* __restrict__ wn,
                                              const T* __restrict__ Nm1, T* __restrict__ N, T* __restrict__ S,
                                              const T* __restrict__ stale, const T* __restrict__ ncorr, T dt, T g, T r)
{
    constexpr int K = KP<T>::value;
    const long sx = d.sx, sy = d.sy;
    const T ylo = stale[0], yhi = stale[1], zlo = stale[2], zhi = stale[3];
    const T kx = T(ph.kap[FC][0]), ky = T(ph.kap[FC][1]), kz = T(ph.kap[FC][2]);
    unsigned l = (unsigned)((j * d.sy + k0) * sizeof(T));
    long o = (long)i * sx + mo;   // uniform; the lane's own offset is l
    Cross<T> st;
    T u1[K];
    st.start(cold, o, l, sx);
    lane_run(un, o, l, u1);
#pragma unroll 1
    for (; i <= ie; i++, o += sx) {
        per_block(l, o);
        // every operand first (one memory round trip), then the arithmetic
        T u0[K], v0[K], v1[K], w[K + 1], nm1[K], nc[K], nv[K], sv[K];
        st.next(cold, o, l, sx, sy);
#pragma unroll
        for (int p = 0; p < K; p++) u0[p] = u1[p];
        lane_run(un, o + sx, l, u1);
        lane_run(vn, o, l, v0);
        lane_run(vn, o + sy, l, v1);
        lane_run(wn, o, l, w);
        // r = 0 (first substage): r N_nm1 is a signed zero, so N_nm1 is not read
        // (the source keeps its value; at most the sign of a zero source differs)
        if (r != T(0)) lane_run(Nm1, o, l, nm1);
        // the learned closure's correction of N (no counterpart in the
        // reference; ncorr is null without a closure)
        if (ncorr) lane_run(ncorr, o, l, nc);
#pragma unroll
        for (int p = 0; p < K; p++) {
            const int k = k0 + p;
            T cx7[7], cy7[7], cz7[7];
            st.at(p, cx7, cy7, cz7);
            const T uval = T(0.5) * (u1[p] + u0[p]), vval = T(0.5) * (v1[p] + v0[p]), wval = T(0.5) * (w[p + 1] + w[p]);
            T nval, diff;
            // A c by the reference's sums (1411-1440, 573-590)
            auto diffusion = [&]() {
                T ax, bx, cx, ay, by, cy, az, bz, cz;
                Visc4<T> none{nullptr, nullptr, nullptr, nullptr};
                coefs<T, FC, 0>(d, ph, none, 0, ax, bx, cx);
                coefs<T, FC, 1>(d, ph, none, 0, ay, by, cy);
                coefs<T, FC, 2>(d, ph, none, 0, az, bz, cz);
                const T axx = ax * cx7[2] + bx * cx7[3] + cx * cx7[4];
                const T axy = ay * cy7[2] + by * cy7[3] + cy * cy7[4];
                const T axz = az * cz7[2] + bz * cz7[3] + cz * cz7[4];
                return axx + axy + axz;
            };
            if constexpr (FAST) {
                T xm, xp, ym, yp, zm, zp;
                const T cx = upwind_term<T>(cx7, i, R.is, R.ie, uval, T(d.dx), T(d.rdx), T(0.0), T(0.0), xm, xp);
                const T cy = upwind_term<T>(cy7, j, R.js, R.je, vval, T(d.dy), T(d.rdy), ylo, yhi, ym, yp);
                const T cz = upwind_term<T>(cz7, k, R.ks, R.ke, wval, T(d.dz), T(d.rdz), zlo, zhi, zm, zp);
                nval = -(cz + cx + cy);
                // FP64: in the reference's roundings.  Where c is 1 up to its last
                // bits the sums leave those bits to rounding, and the front amplifies
                // whatever differs there: with the differences xp - xm, which round
                // less, c departs from the reference by 1.7e-12 in 200 steps at
                // 256x128x128 and 4e-11 in 730 (as the reference does from itself when
                // its initial state changes in the last bit), so by 7e-16.  263.1 ->
                // 263.8 us a launch.
                if constexpr (sizeof(T) == 8) {
                    diff = diffusion();
                } else {
                    diff = kx * (xp - xm);
                    diff = fma(ky, yp - ym, diff);
                    diff = fma(kz, zp - zm, diff);
                }
            } else {
                T D[6];
#pragma unroll
                for (int m = 0; m < 6; m++) D[m] = divh<T>(cx7[m + 1] - cx7[m], T(d.dx), d.rdx);
                const T convx =
                    uval * upwind_d<T>(D, i, R.is, R.ie, uval >= T(0.0) ? 1 : -1, T(d.dx), d.rdx, T(0.0), T(0.0));
#pragma unroll
                for (int m = 0; m < 6; m++) D[m] = divh<T>(cy7[m + 1] - cy7[m], T(d.dy), d.rdy);
                const T convy = vval * upwind_d<T>(D, j, R.js, R.je, vval >= T(0.0) ? 1 : -1, T(d.dy), d.rdy, ylo, yhi);
#pragma unroll
                for (int m = 0; m < 6; m++) D[m] = divh<T>(cz7[m + 1] - cz7[m], T(d.dz), d.rdz);
                const T czd = upwind_d<T>(D, k, R.ks, R.ke, wval >= T(0.0) ? 1 : -1, T(d.dz), d.rdz, zlo, zhi);
                nval = -(wval * czd + convx + convy);
                diff = diffusion();
            }
            if (ncorr) nval += nc[p];
            nv[p] = nval;
            const T conv = (g * nval + r * (r != T(0) ? nm1[p] : T(0)));
            sv[p] = dt * (conv + (g + r) * diff);
        }
        per_block(l, o);
        lane_put(N, o, l, nv, k0, R.ks, R.ke);
        lane_put(S, o, l, sv, k0, R.ks, R.ke);
    }
}

// xmom/ymom/zmom explicit part at the points i .. ie of one (j, k) of
// component F's range: H?_op with mu_old, then the source loop with A(mu_old)
// and the body force (970-989, 1127-1146, 1280-1298).  u, v, w are the old
// velocities; q is the component's own old field.  From plane to plane the x
// stencil, the other components' values and the viscosities that the next
// plane needs again stay in registers: 24 loads a point instead of 37.  Every
// operand of the point is loaded first, so its loads are in flight together;
// the arithmetic below then follows the reference's expressions in its order.
//
// Operands, by component (the "first" and "second" other components):
//   advecting velocity in direction D (1669/1696/1722, 1780/1807/1834,
//   1892/1919/1946): q itself along its own direction, 4-point averages of
//   the others, summed in the order of the offsets below (ao, bo);
//   explicit cross-viscous terms (Hu 1734-1744, Hv 1846-1856, Hw 1958-1970
//   with the live index of 1962): differences of the same 4 values of each
//   other component with the edge viscosities mA (first) and mB (second);
//   A(mu_old) (A_umom/A_vmom/A_wmom, 1443-1536): mu.cell at o - s_F and o
//   along F's own direction, mA and mB along the others.
template <typename T, int F>
__device__ __forceinline__ void coef_vals(const Dims& d, const Phys& ph, int D, T m0, T m1, T& a, T& b, T& c)
{
    const T h = D == 0 ? T(d.dx) : D == 1 ? T(d.dy) : T(d.dz);
    const double rh = D == 0 ? d.rdx : D == 1 ? d.rdy : d.rdz;
    const T del = T(ph.cdel[F][D]);
    a = divh<T>(del * m0, h, rh);
    c = divh<T>(del * m1, h, rh);
    // coefs(): -(a + c) for u along x and y, -a - c otherwise
    b = (F == FU && D != 2) ? -(a + c) : -a - c;
}

template <typename T, int F, bool FAST>
__device__ __forceinline__ void rhs_mom_line(const Dims& d, const Phys& ph, const Rng& R, int i, int ie, int j, int k0,
                                             long mo, const T* __restrict__ u, const T* __restrict__ v,
                                             const T* __restrict__ w, const Visc4<T>& mu, const T* __restrict__ cn,
                                             const T* __restrict__ pg, const T* __restrict__ Nm1,
                                             T* __restrict__ N, T* __restrict__ S, const T* __restrict__ stale,
                                             T dt, T g, T r)
{
    constexpr int K = KP<T>::value;
    const long sx = d.sx, sy = d.sy;
    const long sF = F == FU ? sx : F == FV ? sy : 1;
    const T* __restrict__ q = F == FU ? u : F == FV ? v : w;
    const T* __restrict__ pa = F == FU ? v : u;   // first other component
    const T* __restrict__ pb = F == FW ? v : w;   // second other component
    const T* __restrict__ mA = F == FW ? mu.xz : mu.xy;
    const T* __restrict__ mB = F == FU ? mu.xz : mu.yz;
    unsigned l = (unsigned)((j * d.sy + k0) * sizeof(T));
    const T ylo = stale[0], yhi = stale[1], zlo = stale[2], zhi = stale[3];
    const T kx = T(ph.kap[F][0]), ky = T(ph.kap[F][1]), kz = T(ph.kap[F][2]);
    const T e0 = T(ph.edel[F - FU][0]), e1 = T(ph.edel[F - FU][1]), rRe = T(ph.rRe);
    // c enters only the body force fre (c) of u and v; with fre = 0 that
    // term is a signed zero and the source the same bits without it, so c
    // is not read (the flag is uniform over the launch)
    const bool force = F != FW && ph.fre[F == FU ? 0 : 1] != 0.0;
    const T fre = force ? T(ph.fre[F == FU ? 0 : 1]) : T(0);

    long o = (long)i * sx + mo;   // uniform; the lane's own offset is l
    // Carried along x (as the plane before i would leave them): the stencil;
    // u: v at (j), (j + 1), w at k .. k + K and mu.cell of plane i - 1;
    // v: u at (j - 1), (j) of plane i and mu.xy; w: u at k - 1 .. k + K - 1
    // of plane i and mu.xz.
    Cross<T> st;
    T a1v[K], a2v[K], bw[K + 1], mc[K], ma[K], aw[K + 1];
    st.start(q, o, l, sx);
    if (F == FU) {
        lane_run(pa, o - sx, l, a1v);
        lane_run(pa, o - sx + sy, l, a2v);
        lane_run(pb, o - sx, l, bw);
        lane_run(mu.cell, o - sx, l, mc);
    } else if (F == FV) {
        lane_run(pa, o - sy, l, a1v);
        lane_run(pa, o, l, a2v);
        lane_run(mA, o, l, ma);
    } else {
        lane_run(pa, o - 1, l, aw);
        lane_run(mA, o, l, ma);
    }
#pragma unroll 1
    for (; i <= ie; i++, o += sx) {
        per_block(l, o);
        st.next(q, o, l, sx, sy);
        // the 4-point averages' values and the viscosities of every point, in
        // the reference's order of summation
        T av4[K][4], bv4[K][4], mcs[K][2], mas[K][2], mbs[K][2];
        if (F == FU) {
            // a: -sx, 0, sy, -sx + sy; b: -sx, 0, 1, -sx + 1
            T n1[K], n2[K], nw[K + 1], nc[K], x1[K], x2[K], zw[K + 1];
            lane_run(pa, o, l, n1);
            lane_run(pa, o + sy, l, n2);
            lane_run(pb, o, l, nw);
            lane_run(mu.cell, o, l, nc);
            lane_run(mA, o, l, x1);
            lane_run(mA, o + sy, l, x2);
            lane_run(mB, o, l, zw);
#pragma unroll
            for (int p = 0; p < K; p++) {
                av4[p][0] = a1v[p]; av4[p][1] = n1[p]; av4[p][2] = n2[p]; av4[p][3] = a2v[p];
                bv4[p][0] = bw[p]; bv4[p][1] = nw[p]; bv4[p][2] = nw[p + 1]; bv4[p][3] = bw[p + 1];
                mcs[p][0] = mc[p]; mcs[p][1] = nc[p];
                mas[p][0] = x1[p]; mas[p][1] = x2[p];
                mbs[p][0] = zw[p]; mbs[p][1] = zw[p + 1];
            }
#pragma unroll
            for (int p = 0; p < K; p++) { a1v[p] = n1[p]; a2v[p] = n2[p]; mc[p] = nc[p]; }
#pragma unroll
            for (int p = 0; p <= K; p++) bw[p] = nw[p];
        } else if (F == FV) {
            // a: -sy, sx - sy, 0, sx; b: -sy, -sy + 1, 0, 1
            T n1[K], n2[K], w0[K + 1], w1[K + 1], c0[K], c1[K], na[K], zw[K + 1];
            lane_run(pa, o + sx - sy, l, n1);
            lane_run(pa, o + sx, l, n2);
            lane_run(pb, o - sy, l, w0);
            lane_run(pb, o, l, w1);
            lane_run(mu.cell, o - sy, l, c0);
            lane_run(mu.cell, o, l, c1);
            lane_run(mA, o + sx, l, na);
            lane_run(mB, o, l, zw);
#pragma unroll
            for (int p = 0; p < K; p++) {
                av4[p][0] = a1v[p]; av4[p][1] = n1[p]; av4[p][2] = a2v[p]; av4[p][3] = n2[p];
                bv4[p][0] = w0[p]; bv4[p][1] = w0[p + 1]; bv4[p][2] = w1[p]; bv4[p][3] = w1[p + 1];
                mcs[p][0] = c0[p]; mcs[p][1] = c1[p];
                mas[p][0] = ma[p]; mas[p][1] = na[p];
                mbs[p][0] = zw[p]; mbs[p][1] = zw[p + 1];
            }
#pragma unroll
            for (int p = 0; p < K; p++) { a1v[p] = n1[p]; a2v[p] = n2[p]; ma[p] = na[p]; }
        } else {
            // a: -1, sx - 1, 0, sx; b: -1, 0, sy - 1, sy
            T nw[K + 1], v0[K + 1], v1[K + 1], cw[K + 1], na[K], y0[K], y1[K];
            lane_run(pa, o + sx - 1, l, nw);
            lane_run(pb, o - 1, l, v0);
            lane_run(pb, o + sy - 1, l, v1);
            lane_run(mu.cell, o - 1, l, cw);
            lane_run(mA, o + sx, l, na);
            lane_run(mB, o, l, y0);
            lane_run(mB, o + sy, l, y1);
#pragma unroll
            for (int p = 0; p < K; p++) {
                av4[p][0] = aw[p]; av4[p][1] = nw[p]; av4[p][2] = aw[p + 1]; av4[p][3] = nw[p + 1];
                bv4[p][0] = v0[p]; bv4[p][1] = v0[p + 1]; bv4[p][2] = v1[p]; bv4[p][3] = v1[p + 1];
                mcs[p][0] = cw[p]; mcs[p][1] = cw[p + 1];
                mas[p][0] = ma[p]; mas[p][1] = na[p];
                mbs[p][0] = y0[p]; mbs[p][1] = y1[p];
            }
#pragma unroll
            for (int p = 0; p <= K; p++) aw[p] = nw[p];
#pragma unroll
            for (int p = 0; p < K; p++) ma[p] = na[p];
        }
        T c0v[K], c1v[K], pgs[K], nms[K], nv[K], sv[K];
        if (force) {
            lane_run(cn, o, l, c0v);
            lane_run(cn, o - sF, l, c1v);
        }
        lane_run(pg, o, l, pgs);
        if (r != T(0)) lane_run(Nm1, o, l, nms);   // as in rhs_conc_line
#pragma unroll
        for (int p = 0; p < K; p++) {
            const int k = k0 + p;
            T qx[7], qy[7], qz[7];
            st.at(p, qx, qy, qz);
            const T (&av)[4] = av4[p];
            const T (&bv)[4] = bv4[p];
            const T mc0 = mcs[p][0], mc1 = mcs[p][1], ma0 = mas[p][0], ma1 = mas[p][1], mb0 = mbs[p][0], mb1 = mbs[p][1];
            const T cn0 = force ? c0v[p] : T(0), cn1 = force ? c1v[p] : T(0);
            const T pgv = pgs[p], nm1 = r != T(0) ? nms[p] : T(0);

            const T alpha = g + r;
            const T vx = F == FU ? qx[3] : T(0.25) * (av[0] + av[1] + av[2] + av[3]);
            const T vy = F == FV ? qy[3] : F == FU ? T(0.25) * (av[0] + av[1] + av[2] + av[3])
                                                   : T(0.25) * (bv[0] + bv[1] + bv[2] + bv[3]);
            const T vz = F == FW ? qz[3] : T(0.25) * (bv[0] + bv[1] + bv[2] + bv[3]);
            // the cross-viscous differences at the upper and lower edges
            const T a1 = F == FU ? av[2] - av[3] : av[3] - av[1];
            const T a0 = F == FU ? av[1] - av[0] : av[2] - av[0];
            const T b1 = F == FU ? bv[2] - bv[3] : F == FV ? bv[3] - bv[1] : bv[3] - bv[2];
            const T b0 = F == FV ? bv[2] - bv[0] : bv[1] - bv[0];
            // mu below and above the point along x, y and z
            const T mx0 = F == FU ? mc0 : ma0, mx1 = F == FU ? mc1 : ma1;
            const T my0 = F == FU ? ma0 : F == FV ? mc0 : mb0, my1 = F == FU ? ma1 : F == FV ? mc1 : mb1;
            const T mz0 = F == FW ? mc0 : mb0, mz1 = F == FW ? mc1 : mb1;
            const T Re = T(ph.Re);
            if constexpr (FAST) {
                T xm, xp, ym, yp, zm, zp;
                const T cx = upwind_term<T>(qx, i, R.is, R.ie, vx, T(d.dx), T(d.rdx), T(0.0), T(0.0), xm, xp);
                const T cy = upwind_term<T>(qy, j, R.js, R.je, vy, T(d.dy), T(d.rdy), ylo, yhi, ym, yp);
                const T cz = upwind_term<T>(qz, k, R.ks, R.ke, vz, T(d.dz), T(d.rdz), zlo, zhi, zm, zp);
                T nval = fma(e0, fma(ma1, a1, -(ma0 * a0)), -(cz + cx + cy));
                nval = fma(e1, fma(mb1, b1, -(mb0 * b0)), nval);
                nv[p] = nval;
                T visc = kx * fma(mx1, xp, -(mx0 * xm));
                visc = fma(ky, fma(my1, yp, -(my0 * ym)), visc);
                visc = fma(kz, fma(mz1, zp, -(mz0 * zm)), visc);
                visc = fma(-rRe, pgv, visc);
                if (force) visc = fma(-fre, T(0.5) * (cn0 + cn1), visc);
                sv[p] = dt * fma(alpha, visc, fma(g, nval, r * nm1));
            } else {
                // convec_term: upwind derivatives along x, y, z
                T D[6];
#pragma unroll
                for (int m = 0; m < 6; m++) D[m] = divh<T>(qx[m + 1] - qx[m], T(d.dx), d.rdx);
                const T convx = vx * upwind_d<T>(D, i, R.is, R.ie, vx >= T(0.0) ? 1 : -1, T(d.dx), d.rdx, T(0.0), T(0.0));
#pragma unroll
                for (int m = 0; m < 6; m++) D[m] = divh<T>(qy[m + 1] - qy[m], T(d.dy), d.rdy);
                const T convy = vy * upwind_d<T>(D, j, R.js, R.je, vy >= T(0.0) ? 1 : -1, T(d.dy), d.rdy, ylo, yhi);
#pragma unroll
                for (int m = 0; m < 6; m++) D[m] = divh<T>(qz[m + 1] - qz[m], T(d.dz), d.rdz);
                const T dzd = upwind_d<T>(D, k, R.ks, R.ke, vz >= T(0.0) ? 1 : -1, T(d.dz), d.rdz, zlo, zhi);
                const T ct = vz * dzd + convx + convy;
                // explicit_n: -convec_term + the cross-viscous terms, left to right
                const T p1 = e0 * ma1 * a1, m1 = e0 * ma0 * a0;
                const T p2 = e1 * mb1 * b1, m2 = e1 * mb0 * b0;
                const T nval = -ct + p1 - m1 + p2 - m2;
                nv[p] = nval;
                // source: dt [g N + r N_nm1 + alpha A(mu_old) q + alpha (body force)]
                T ax, bx, cx, ay, by, cy, az, bz, cz;
                coef_vals<T, F>(d, ph, 0, mx0, mx1, ax, bx, cx);
                coef_vals<T, F>(d, ph, 1, my0, my1, ay, by, cy);
                coef_vals<T, F>(d, ph, 2, mz0, mz1, az, bz, cz);
                const T conv = (g * nval + r * nm1);
                const T axx = ax * qx[2] + bx * qx[3] + cx * qx[4];
                const T axy = ay * qy[2] + by * qy[3] + cy * qy[4];
                const T axz = az * qz[2] + bz * qz[3] + cz * qz[4];
                const T visc = alpha * (axx + axy + axz);
                T bodyforce;
                if (!force) bodyforce = alpha * (-divh<T>(pgv, Re, ph.rRe));
                else bodyforce = alpha * (-fre * (T(0.5) * (cn0 + cn1)) - divh<T>(pgv, Re, ph.rRe));
                sv[p] = dt * (conv + visc + bodyforce);
            }
        }
        per_block(l, o);
        lane_put(N, o, l, nv, k0, R.ks, R.ke);
        lane_put(S, o, l, sv, k0, R.ks, R.ke);
    }
}

// the explicit parts of n fields (F: FC, FU, FV or FW) in one launch: np
// planes a thread, the fields' blocks of the same planes next to each other in
// dispatch order, so that the velocities and viscosities which they share
// come from HBM once and a small grid pays for one launch: at 256x128x128
// FP64 one launch per component moved 9.8 fields and the concentration's 6.9,
// together 36, the joint one moves 25 (there are 23).  us, four launches ->
// one: 256x128x128 FP64 369 -> 263, mixed 169 -> 134; 512x256x256 FP64 2740 ->
// 1920, mixed 1210 -> 1000; 64x32x32 FP64 20 -> 9.  FP32 is bound by vector issue (92% of the cycles);
// FP64 by latency with two waves per vector unit (54% issue, 36% waiting).
template <typename T>
struct RhsSets {
    int n;
    struct { int F; const T* pg; const T* Nm1; T* N; T* S; } s[4];
};
template <typename T, bool FAST, bool B = false>
__global__ __launch_bounds__(256, sizeof(T) == 8 ? 2 : 6) void k_rhs(Dims d, Phys ph0, RhsSets<T> rs, const T* __restrict__ cold,
                                             const T* __restrict__ u, const T* __restrict__ v, const T* __restrict__ w,
                                             Visc4<T> mu, const T* __restrict__ cn, const T* __restrict__ ncorr,
                                             const T* __restrict__ stale0, const double* __restrict__ scal, T g, T r,
                                             int np, Bt bt)
{
    const int2 tl = xcd_tile();
    const int k = (tl.x * blockDim.x + threadIdx.x) * KP<T>::value + 1;
    const int j = tl.y * blockDim.y + threadIdx.y + 1;
    int il;
    const int m = bt_member(bt, blockIdx.z, gridDim.z, il);
    const int grp = il / rs.n, q = il - grp * rs.n;
    const auto& s = rs.s[q];
    const int F = s.F;
    const Rng R = field_rng(d, F);
    const int i0 = 3 + grp * np, i = max(i0, R.is), ie = min(i0 + np - 1, R.ie);
    if (k + KP<T>::value <= R.ks || k > R.ke || j < R.js || j > R.je) return;
    const Phys& ph = bt_phys<B>(bt, ph0, m);
    const T* stale = stale0 + m * 16 + 4 * F;
    const T dt = T(scal[m * S_SIZE + S_DT]);
    const long mo = m * bt.fs;
    if (F == FC)
        rhs_conc_line<T, FAST>(d, ph, R, i, ie, j, k, mo, cold, u, v, w, s.Nm1, s.N, s.S, stale, ncorr, dt, g, r);
    else if (F == FU)
        rhs_mom_line<T, FU, FAST>(d, ph, R, i, ie, j, k, mo, u, v, w, mu, cn, s.pg, s.Nm1, s.N, s.S, stale, dt, g, r);
    else if (F == FV)
        rhs_mom_line<T, FV, FAST>(d, ph, R, i, ie, j, k, mo, u, v, w, mu, cn, s.pg, s.Nm1, s.N, s.S, stale, dt, g, r);
    else
        rhs_mom_line<T, FW, FAST>(d, ph, R, i, ie, j, k, mo, u, v, w, mu, cn, s.pg, s.Nm1, s.N, s.S, stale, dt, g, r);
}

// --------------------------------------------------------- line solvers
//
// The implicit sweeps of concentration (592-698) and xmom/ymom/zmom
// (992-1102, 1149-1255, 1301-1403): tridiag_1rhs (3511-3536) on y- and
// z-lines, pll_tridiag at one rank (pll_tridiag.c:21-47, 96-110) on x-lines,
// for (I - fac A) with fac = dt*alpha/2 and the field's boundary rows.
//
// One thread per line.  A row's upper coefficient c is the same expression
// as the next row's lower coefficient a (e.g. A_umom 1460-1461: xy[j+1] vs
// xy[j] of the next row), so each row loads one viscosity value.  Rows are
// loaded LB at a time, one batch ahead of the recurrence, so memory latency
// overlaps the serial elimination.  The Thomas factors go to the scratch
// field CC; the solution overwrites S in place.

// rows prefetched per batch: x-lines are the fewest (one wave per SIMD),
// so they get the deepest prefetch
template <int DIR> struct LinePrefetch { static constexpr int value = DIR == 0 ? 16 : 8; };

// one field's lines in one direction
template <typename T>
struct LineSet {
    T* S;                 // source in, solution out
    T* CC;                // Thomas factors
    const T* mu;          // viscosity of the lower coefficient of row 0 + x*stride, or nullptr
    long mu_off;          // offset of that value from the row's own point
    T del, h;             // coefficient = del*mu/h (A_*mom 1453-1532)
    double rh;            // 1/h rounded on the host (divh)
    T ca, cb, cc;         // constant coefficients when mu == nullptr (A_conc)
    int bc0, bc1;         // boundary kinds of the first and last row (x: first only)
    Rng R;
    // x-lines only: the update q_new = q_old + delta and the outflow face
    const T* qold;
    T* qnew;
    T* N;
    const T* Nm1;
    int ghost_c;          // also fill c_new's y/z ghosts (700-712)
    int ghost_v;          // 0, or FU/FV/FW: also fill that component's ghosts (velo_ghost_point)
    int jg, kg, inlet;    // which those are: y ghosts, z ghosts, inlet ghosts
    int F;                // the field (FC, FU, FV, FW): its constants in a batch's table
};

// member m's copy of a line set in a batched launch: the fields moved to
// the member's, the constant coefficients from the batch's table
// [m][F][DIR][del, ca, cb, cc] (the host's values for that member)
template <typename T, int DIR>
__device__ __forceinline__ LineSet<T> bt_lines(const Bt& bt, const LineSet<T>& L0, int m)
{
    LineSet<T> L = L0;
    if (bt.nm == 1) return L;
    L.S = bt_f(bt, L.S, m);
    L.CC = bt_f(bt, L.CC, m);
    L.mu = bt_f(bt, L.mu, m);
    L.qold = bt_f(bt, L.qold, m);
    L.qnew = bt_f(bt, L.qnew, m);
    L.N = bt_f(bt, L.N, m);
    L.Nm1 = bt_f(bt, L.Nm1, m);
    const T* k = reinterpret_cast<const T*>(bt.lc) + ((m * 4 + L.F) * 3 + DIR) * 4;
    L.del = k[0];
    L.ca = k[1];
    L.cb = k[2];
    L.cc = k[3];
    return L;
}

template <typename T>
struct LineSets {
    LineSet<T> s[3];
};

// The ghost copies of update_velo_boundary / update_veloghost_points
// (2701-2755, 2810-2885; k_velo_ghost) whose source is the new value q of
// component F at interior point (i, j, k): z ghosts of u and v (copies),
// y ghosts of u and w (negated), inlet ghosts of v and w (negated).  The
// fused step writes them where q is written; ghost sources a step never
// rewrites (u at the inlet face, v at the bottom wall, w at the side wall)
// keep the ghosts they were given at set-up.
template <typename T>
__device__ __forceinline__ void velo_ghost_point(const Dims& d, int F, T* __restrict__ p, int i, int j, int k, T val)
{
    // p points at (i, j, k); i is in [3, nx + 2] for every caller
    if (F != FW) {
        if (k == 1) p[-1] = val;
        if (k == d.nz) p[1] = val;
    }
    if (F != FV) {
        if (j == 1) p[-d.sy] = -val;
        if (j == d.ny) p[d.sy] = -val;
    }
    if (F != FU && i == 3) p[-d.sx] = -val;
}

template <typename T, int DIR>
__global__ __launch_bounds__(256) void k_sweep(Dims d, LineSets<T> sets, const double* __restrict__ scal, int slot,
                                               T g, T r)
{
    constexpr int LB = LinePrefetch<DIR>::value;
    const LineSet<T>& L = sets.s[blockIdx.y];
    const Rng R = L.R;
    // lines: DIR 0 (x) over (j,k), DIR 1 (y) over (i,k), DIR 2 (z) over (i,j);
    // the fastest line index runs over k for x and y (coalesced)
    const int n0 = DIR == 2 ? R.je - R.js + 1 : R.ke - R.ks + 1;
    const int n1 = DIR == 0 ? R.je - R.js + 1 : R.ie - R.is + 1;
    const long l = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= (long)n0 * n1) return;
    const int a0 = (int)(l % n0), a1 = (int)(l / n0);
    int i, j, k, n;
    long st;
    if (DIR == 0) { k = R.ks + a0; j = R.js + a1; i = R.is; n = R.ie - R.is + 1; st = d.sx; }
    else if (DIR == 1) { k = R.ks + a0; i = R.is + a1; j = R.js; n = R.je - R.js + 1; st = d.sy; }
    else { j = R.js + a0; i = R.is + a1; k = R.ks; n = R.ke - R.ks + 1; st = 1; }
    const long o0 = IX(d, i, j, k);
    T* __restrict__ S = L.S + o0;
    T* __restrict__ CC = L.CC + o0;
    const bool cst = L.mu == nullptr;
    const T* __restrict__ mu = cst ? nullptr : L.mu + o0 + L.mu_off;
    const T del = L.del, h = L.h;
    const double rh = L.rh;
    const T dt = T(scal[S_DT]);
    const T fac = T(0.5) * dt * (g + r);
    const T zero = T(0.0);

    T bcor = T(0.0);
    if (DIR == 0) {
        // explicit outflow face iend+1 (677-683 and matching lines)
        const long ob = o0 + (long)n * st;
        const T vbulk = T(scal[S_RK + 4 * slot]);
        const T nb = divh<T>(-vbulk * (L.qold[ob] - L.qold[ob - st]), T(d.dx), d.rdx);
        L.N[ob] = nb;
        bcor = dt * (g * nb + r * L.Nm1[ob]);
        L.qnew[ob] = L.qold[ob] + bcor;
    }

    // ---- forward elimination
    T araw = cst ? L.ca : divh<T>(del * mu[0], h, rh);
    T pc = T(0.0), pr = T(0.0);
    T cs[LB], cm[LB], ns[LB], nm[LB];
#pragma unroll
    for (int t = 0; t < LB; t++) {
        if (t < n) { cs[t] = S[(long)t * st]; if (!cst) cm[t] = mu[(long)(t + 1) * st]; }
    }
    for (int x0 = 0; x0 < n; x0 += LB) {
#pragma unroll
        for (int t = 0; t < LB; t++) {
            const int x = x0 + LB + t;
            if (x < n) { ns[t] = S[(long)x * st]; if (!cst) nm[t] = mu[(long)(x + 1) * st]; }
        }
#pragma unroll
        for (int t = 0; t < LB; t++) {
            const int x = x0 + t;
            if (x < n) {
                const T craw = cst ? L.cc : divh<T>(del * cm[t], h, rh);
                const T braw = cst ? L.cb : -(araw + craw);
                const T a = -fac * araw;
                T b = T(1.0) - fac * braw;
                T c = -fac * craw;
                T rhs = cs[t];
                if (x == 0) apply_bc(L.bc0, b, a, rhs);
                if (DIR == 0) {
                    if (x == n - 1) rhs -= c * bcor;
                    if (x == 0) { b = b - zero * a; c = c / b; rhs = (rhs - zero * a) / b; }
                    else { b = (b - pc * a); c = c / b; rhs = (rhs - pr * a) / b; }
                } else {
                    if (x == n - 1) apply_bc(L.bc1, b, c, rhs);
                    T bb;
                    if (x == 0) { bb = b; c = c / bb; rhs = rhs / bb; }
                    else { bb = b - pc * a; c = c / bb; rhs = (rhs - pr * a) / bb; }
                }
                CC[(long)x * st] = c;
                S[(long)x * st] = rhs;
                pc = c; pr = rhs;
                araw = craw;
            }
        }
#pragma unroll
        for (int t = 0; t < LB; t++) { cs[t] = ns[t]; cm[t] = nm[t]; }
    }

    // ---- back substitution (row n-1 is final already)
    if (DIR == 0) {
        pr = pr - pc * zero;
        L.qnew[o0 + (long)(n - 1) * st] = L.qold[o0 + (long)(n - 1) * st] + pr;
    }
    T bs[LB], bc[LB], bq[LB], qs[LB], qc[LB], qq[LB];
#pragma unroll
    for (int t = 0; t < LB; t++) {
        const int x = n - 2 - t;
        if (x >= 0) {
            bs[t] = S[(long)x * st]; bc[t] = CC[(long)x * st];
            if (DIR == 0) bq[t] = L.qold[o0 + (long)x * st];
        }
    }
    for (int x0 = n - 2; x0 >= 0; x0 -= LB) {
#pragma unroll
        for (int t = 0; t < LB; t++) {
            const int x = x0 - LB - t;
            if (x >= 0) {
                qs[t] = S[(long)x * st]; qc[t] = CC[(long)x * st];
                if (DIR == 0) qq[t] = L.qold[o0 + (long)x * st];
            }
        }
#pragma unroll
        for (int t = 0; t < LB; t++) {
            const int x = x0 - t;
            if (x >= 0) {
                T rr;
                if (DIR == 0) {
                    rr = bs[t] - bc[t] * pr;
                    L.qnew[o0 + (long)x * st] = bq[t] + rr;
                } else {
                    rr = bs[t] - pr * bc[t];
                    S[(long)x * st] = rr;
                }
                pr = rr;
            }
        }
#pragma unroll
        for (int t = 0; t < LB; t++) { bs[t] = qs[t]; bc[t] = qc[t]; bq[t] = qq[t]; }
    }

    if (DIR == 0 && L.ghost_v) {
        T* qn = L.qnew;
        for (int ii = R.is; ii <= R.ie; ii++) {
            T* p = qn + IX(d, ii, j, k);
            velo_ghost_point<T>(d, L.ghost_v, p, ii, j, k, *p);
        }
    }
    if (DIR == 0 && L.ghost_c) {
        // ghost copies of this line's values: y ghosts (701-704), then z
        // ghosts incl. the y-ghost rows (707-712)
        T* qn = L.qnew;
        for (int ii = R.is; ii <= R.ie; ii++) {
            const T val = qn[IX(d, ii, j, k)];
            if (j == R.js) qn[IX(d, ii, j - 1, k)] = val;
            if (j == R.je) qn[IX(d, ii, j + 1, k)] = val;
            if (k == R.ks) {
                qn[IX(d, ii, j, k - 1)] = val;
                if (j == R.js) qn[IX(d, ii, j - 1, k - 1)] = val;
                if (j == R.je) qn[IX(d, ii, j + 1, k - 1)] = val;
            }
            if (k == R.ke) {
                qn[IX(d, ii, j, k + 1)] = val;
                if (j == R.js) qn[IX(d, ii, j - 1, k + 1)] = val;
                if (j == R.je) qn[IX(d, ii, j + 1, k + 1)] = val;
            }
        }
    }
}

// z-lines through LDS.  Rows along k are contiguous in memory, so a
// thread-per-line sweep would make every load of a wavefront touch 64
// different cache lines.  Here a block of 64 threads owns 64 z-lines (one i,
// 64 consecutive j) and moves their rows through LDS in chunks of ZC rows:
// ZC/2 threads read one line's chunk as 16-byte pieces (whole cache lines),
// the next chunk is fetched into registers while the current one is solved
// from LDS.  Arithmetic identical to k_sweep<T, 2>.
constexpr int ZC = 16;
constexpr int ZL = 64;

template <typename T>
__global__ __launch_bounds__(ZL) void k_sweep_z_lds(Dims d, LineSets<T> sets, const double* __restrict__ scal, T g,
                                                    T r)
{
    __shared__ T sS[ZL][ZC + 1];
    __shared__ T sA[ZL][ZC + 1];   // viscosity in, Thomas factors out
    const LineSet<T>& L = sets.s[blockIdx.z];
    const Rng R = L.R;
    const int nj = R.je - R.js + 1, n = R.ke - R.ks + 1;
    const int i = R.is + blockIdx.y;
    if (i > R.ie) return;
    const int j0 = R.js + blockIdx.x * ZL;
    const int nl = min(ZL, nj - (int)(blockIdx.x * ZL));
    if (nl <= 0) return;
    const int t = threadIdx.x;
    const bool mine = t < nl;
    const long base = IX(d, i, j0, R.ks);   // row 0 of line 0; line q at base + q*sy
    const bool cst = L.mu == nullptr;
    const T* __restrict__ mu = cst ? nullptr : L.mu + L.mu_off;
    const T del = L.del, h = L.h;
    const double rh = L.rh;
    const T fac = T(0.5) * T(scal[S_DT]) * (g + r);
    // cooperative chunk copy: element e of the chunk = (line e / ZC, row e % ZC)
    constexpr int PER = ZL * ZC / ZL;   // elements per thread per chunk
    T rs[PER], rm[PER];
    auto gload = [&](int k0) {
#pragma unroll
        for (int p = 0; p < PER; p++) {
            const int e = p * ZL + t, q = e / ZC, kk = e % ZC;
            const long o = base + (long)q * d.sy + k0 + kk;
            if (q < nl && k0 + kk < n) {
                rs[p] = L.S[o];
                if (!cst) rm[p] = mu[o + 1];
            }
        }
    };
    auto sstore = [&]() {
#pragma unroll
        for (int p = 0; p < PER; p++) {
            const int e = p * ZL + t, q = e / ZC, kk = e % ZC;
            sS[q][kk] = rs[p];
            if (!cst) sA[q][kk] = rm[p];
        }
    };
    auto gstore = [&](int k0, bool with_cc) {
#pragma unroll
        for (int p = 0; p < PER; p++) {
            const int e = p * ZL + t, q = e / ZC, kk = e % ZC;
            const long o = base + (long)q * d.sy + k0 + kk;
            if (q < nl && k0 + kk < n) {
                L.S[o] = sS[q][kk];
                if (with_cc) L.CC[o] = sA[q][kk];
            }
        }
    };

    // ---- forward elimination
    T araw = cst ? L.ca : (mine ? divh<T>(del * mu[base + (long)t * d.sy], h, rh) : T(0.0));
    T pc = T(0.0), pr = T(0.0);
    gload(0);
    for (int k0 = 0; k0 < n; k0 += ZC) {
        __syncthreads();
        sstore();
        __syncthreads();
        if (k0 + ZC < n) gload(k0 + ZC);
        if (mine) {
            const int m = min(ZC, n - k0);
            for (int kk = 0; kk < m; kk++) {
                const int x = k0 + kk;
                const T craw = cst ? L.cc : divh<T>(del * sA[t][kk], h, rh);
                const T braw = cst ? L.cb : -(araw + craw);
                const T a = -fac * araw;
                T b = T(1.0) - fac * braw;
                T c = -fac * craw;
                T rhs = sS[t][kk];
                if (x == 0) apply_bc(L.bc0, b, a, rhs);
                if (x == n - 1) apply_bc(L.bc1, b, c, rhs);
                T bb;
                if (x == 0) { bb = b; c = c / bb; rhs = rhs / bb; }
                else { bb = b - pc * a; c = c / bb; rhs = (rhs - pr * a) / bb; }
                sA[t][kk] = c;
                sS[t][kk] = rhs;
                pc = c; pr = rhs;
                araw = craw;
            }
        }
        __syncthreads();
        gstore(k0, true);
    }
    // ---- back substitution, chunks from the end; pr = solution of row n-1
    const int last0 = ((n - 1) / ZC) * ZC;
    for (int k0 = last0; k0 >= 0; k0 -= ZC) {
        __syncthreads();
#pragma unroll
        for (int p = 0; p < PER; p++) {
            const int e = p * ZL + t, q = e / ZC, kk = e % ZC;
            const long o = base + (long)q * d.sy + k0 + kk;
            if (q < nl && k0 + kk < n) { sS[q][kk] = L.S[o]; sA[q][kk] = L.CC[o]; }
        }
        __syncthreads();
        if (mine) {
            const int m = min(ZC, n - k0);
            for (int kk = m - 1; kk >= 0; kk--) {
                const int x = k0 + kk;
                if (x == n - 1) continue;
                const T rr = sS[t][kk] - pr * sA[t][kk];
                sS[t][kk] = rr;
                pr = rr;
            }
        }
        __syncthreads();
        gstore(k0, false);
    }
}

// ------------------------------------------------------------ viscosity

// calculate_viscosity (843-886) / calculate_viscosity_nmvp (889-948): cell
// centres on a one-cell ring, and edges from the 4-point mean of c (mean
// first, then the law).
//
// A (j, k) plane (j 0 .. ny+1, k 0 .. nz+1) is cut into chunks of 256 lanes,
// one per block, of rows of nz + 2 lanes (k = 1 .. nz+1, then 0; no lane idle,
// for the exponentials are half its time in FP64); gridDim.x (chunks per plane) is a
// multiple of 8 so that the
// XCD a block runs on (its linear id mod 8) depends only on blockIdx.x, and
// XCD x takes chunks x nb/8 .. (x+1) nb/8 - 1 of every plane: the previous
// plane's c (o - sx) was read into the same XCD's L2.
template <typename T, bool B = false>
__global__ __launch_bounds__(256) void k_visc(Dims d, Phys ph0, const T* __restrict__ cn, T* __restrict__ cell,
                                              T* __restrict__ xy, T* __restrict__ xz, T* __restrict__ yz, Bt bt)
{
    // member: blockIdx.z
    const int m = blockIdx.z;
    const Phys& ph = bt_phys<B>(bt, ph0, m);
    cn = bt_f(bt, cn, m);
    cell = bt_f(bt, cell, m);
    xy = bt_f(bt, xy, m);
    xz = bt_f(bt, xz, m);
    yz = bt_f(bt, yz, m);
    const int nb8 = gridDim.x >> 3;
    const int chunk = (blockIdx.x & 7) * nb8 + (blockIdx.x >> 3);
    const int l = chunk * 256 + threadIdx.x;
    const int w = d.nz + 2;
    const int j = l / w, a = l - j * w;                        // 0 .. ny+1
    if (j > d.ny + 1) return;
    const int k = a <= d.nz ? a + 1 : 0;                       // 1 .. nz+1, 0
    const int i = blockIdx.y + 2;                              // 2 .. nx+3
    const long o = IX(d, i, j, k), sx = d.sx, sy = d.sy;
    // the seven values first (all inside the array: i >= 2 leaves a ghost
    // plane below o - sx - sy - 1), then the laws
    const T c0 = cn[o], cxm = cn[o - sx], cym = cn[o - sy], czm = cn[o - 1];
    const T cxy = cn[o - sx - sy], cxz = cn[o - sx - 1], cyz = cn[o - sy - 1];
    cell[o] = visc_law<T>(ph, c0);
    const bool ix = i >= 3, iy = j >= 1, iz = k >= 1;
    const bool jx = j <= d.ny, kx = k <= d.nz, ii = i <= d.nx + 2;
    if (ix && iy && kx && iz) xy[o] = visc_law<T>(ph, T(0.25) * (cxy + cym + cxm + c0));
    if (ix && iy && jx && iz) xz[o] = visc_law<T>(ph, T(0.25) * (cxz + czm + cxm + c0));
    if (ix && ii && iy && iz) yz[o] = visc_law<T>(ph, T(0.25) * (cyz + czm + cym + c0));
}

// ----------------------------------------------------------- ghost rules

// update_velo_boundary (2701-2755) == update_veloghost_points (2810-2885)
// at one rank.  Three disjoint sets: z ghosts of u,v; y ghosts of u,w;
// inlet ghosts of v,w.
template <typename T>
__global__ void k_velo_ghost(Dims d, T* __restrict__ u, T* __restrict__ v, T* __restrict__ w)
{
    const int nA = d.nx * d.ny, nB = d.nx * d.nz, nC = d.ny * d.nz;
    int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l < nA) {
        const int i = 3 + l / d.ny, j = 1 + l % d.ny;
        const long lo = IX(d, i, j, 0), hi = IX(d, i, j, d.nz + 1);
        u[lo] = u[lo + 1]; v[lo] = v[lo + 1];
        u[hi] = u[hi - 1]; v[hi] = v[hi - 1];
        return;
    }
    l -= nA;
    if (l < nB) {
        const int i = 3 + l / d.nz, k = 1 + l % d.nz;
        const long lo = IX(d, i, 0, k), hi = IX(d, i, d.ny + 1, k);
        u[lo] = -u[lo + d.sy]; w[lo] = -w[lo + d.sy];
        u[hi] = -u[hi - d.sy]; w[hi] = -w[hi - d.sy];
        return;
    }
    l -= nB;
    if (l < nC) {
        const int j = 1 + l / d.nz, k = 1 + l % d.nz;
        const long lo = IX(d, 2, j, k);
        v[lo] = -v[lo + d.sx]; w[lo] = -w[lo + d.sx];
    }
}

// update_phi_ghosts (2758-2807): Neumann on every face.
template <typename T>
__global__ void k_phi_ghost(Dims d, T* __restrict__ phi)
{
    const int nA = d.nx * d.ny, nB = d.nx * d.nz, nC = d.ny * d.nz;
    int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l < nA) {
        const int i = 3 + l / d.ny, j = 1 + l % d.ny;
        const long lo = IX(d, i, j, 0), hi = IX(d, i, j, d.nz + 1);
        phi[lo] = phi[lo + 1]; phi[hi] = phi[hi - 1];
        return;
    }
    l -= nA;
    if (l < nB) {
        const int i = 3 + l / d.nz, k = 1 + l % d.nz;
        const long lo = IX(d, i, 0, k), hi = IX(d, i, d.ny + 1, k);
        phi[lo] = phi[lo + d.sy]; phi[hi] = phi[hi - d.sy];
        return;
    }
    l -= nB;
    if (l < nC) {
        const int j = 1 + l / d.nz, k = 1 + l % d.nz;
        const long lo = IX(d, 2, j, k), hi = IX(d, d.nx + 3, j, k);
        phi[lo] = phi[lo + d.sx]; phi[hi] = phi[hi - d.sx];
    }
}

// ------------------------------------------------------------ projection

// divergence (1983-1999).  Writes div (if non-null) and/or the scaled
// Poisson source Re/(dt*alpha)*div packed as [x][y][z] (2018-2024).
template <typename T>
__global__ __launch_bounds__(256) void k_div(Dims d, Phys ph, const T* __restrict__ u, const T* __restrict__ v,
                                             const T* __restrict__ w, T* __restrict__ div, T* __restrict__ P,
                                             const double* __restrict__ scal, T g, T r)
{
    const int2 tl = xcd_tile();
    const int k = tl.x * blockDim.x + threadIdx.x + 1;
    const int j = tl.y * blockDim.y + threadIdx.y + 1;
    const int i = blockIdx.z + 3;
    if (k > d.nz || j > d.ny) return;
    const long o = IX(d, i, j, k);
    const T dvx = divh<T>(u[o + d.sx] - u[o], T(d.dx), d.rdx);
    const T dvy = divh<T>(v[o + d.sy] - v[o], T(d.dy), d.rdy);
    const T dvz = divh<T>(w[o + 1] - w[o], T(d.dz), d.rdz);
    const T dv = (dvx + dvy + dvz);
    if (div) div[o] = dv;
    if (P) {
        const T fac = T(ph.Re) / (T(scal[S_DT]) * (g + r));
        P[((long)(i - 3) * d.ny + (j - 1)) * d.nz + (k - 1)] = fac * dv;
    }
}

// phisolver_dct packing of an existing div field (2016-2024)
template <typename T>
__global__ __launch_bounds__(256) void k_pack_div(Dims d, Phys ph, const T* __restrict__ div, T* __restrict__ P,
                                                  const double* __restrict__ scal, T g, T r)
{
    const int2 bt = xcd_tile();
    const int k = bt.x * blockDim.x + threadIdx.x + 1;
    const int j = bt.y * blockDim.y + threadIdx.y + 1;
    const int i = blockIdx.z + 3;
    if (k > d.nz || j > d.ny) return;
    const T fac = T(ph.Re) / (T(scal[S_DT]) * (g + r));
    P[((long)(i - 3) * d.ny + (j - 1)) * d.nz + (k - 1)] = fac * div[IX(d, i, j, k)];
}

// Per-mode x-line solve of the Poisson problem in (y,z) DCT space
// (2037-2091): a = c = 1/dx^2, b = -2/dx^2 + lam_y + lam_z, Neumann at the
// inlet; at the outlet Neumann except mode (0,0), whose ghost phi is the
// constant 0.  One thread per mode, coalesced over kz; in place.
// one mode's x-line in arithmetic type U on fields of type T
template <typename U, typename T>
__device__ __forceinline__ void pois_line(const Dims& d, U ly, U lz, int jy, int kz, long l, T* __restrict__ P,
                                          T* __restrict__ CC)
{
    constexpr int PB = 16;   // rows prefetched per batch
    const long nm = (long)d.ny * d.nz;
    const int n = d.nx;
    const U dx2i = U(1.0) / (U(d.dx) * U(d.dx));
    const U phiconst = U(0.0), zero = U(0.0);
    const U bmid = U(-2.0) * dx2i + ly + lz;
    T* __restrict__ p = P + l;
    T* __restrict__ cq = CC + l;
    U pc = U(0.0), pr = U(0.0);
    U cur[PB], nxt[PB];
#pragma unroll
    for (int t = 0; t < PB; t++) if (t < n) cur[t] = U(p[(long)t * nm]);
    for (int x0 = 0; x0 < n; x0 += PB) {
#pragma unroll
        for (int t = 0; t < PB; t++) if (x0 + PB + t < n) nxt[t] = U(p[(long)(x0 + PB + t) * nm]);
#pragma unroll
        for (int t = 0; t < PB; t++) {
            const int x = x0 + t;
            if (x < n) {
                const U a = dx2i;
                U b = bmid, c = dx2i, rhs = cur[t];
                if (x == 0) b += a;
                if (x == n - 1) {
                    if (jy == 0 && kz == 0) rhs -= c * phiconst;
                    else b += c;
                }
                if (x == 0) { b = b - zero * a; c = c / b; rhs = (rhs - zero * a) / b; }
                else { b = (b - pc * a); c = c / b; rhs = (rhs - pr * a) / b; }
                cq[(long)x * nm] = T(c);
                p[(long)x * nm] = T(rhs);
                pc = c; pr = rhs;
            }
        }
#pragma unroll
        for (int t = 0; t < PB; t++) cur[t] = nxt[t];
    }
    pr = pr - pc * zero;
    p[(long)(n - 1) * nm] = T(pr);
    U cs[PB], cc[PB], ns[PB], nc[PB];
#pragma unroll
    for (int t = 0; t < PB; t++) { const int x = n - 2 - t; if (x >= 0) { cs[t] = U(p[(long)x * nm]); cc[t] = U(cq[(long)x * nm]); } }
    for (int x0 = n - 2; x0 >= 0; x0 -= PB) {
#pragma unroll
        for (int t = 0; t < PB; t++) {
            const int x = x0 - PB - t;
            if (x >= 0) { ns[t] = U(p[(long)x * nm]); nc[t] = U(cq[(long)x * nm]); }
        }
#pragma unroll
        for (int t = 0; t < PB; t++) {
            const int x = x0 - t;
            if (x >= 0) {
                const U rr = cs[t] - cc[t] * pr;
                p[(long)x * nm] = T(rr);
                pr = rr;
            }
        }
#pragma unroll
        for (int t = 0; t < PB; t++) { cs[t] = ns[t]; cc[t] = nc[t]; }
    }
}

// The (0,0) pencil (the mean of every x-plane, closed by the ghost phi = 0
// at the outlet) is solved in FP64 whatever the field type: it is the
// gauge of the otherwise singular Neumann problem and carries the most
// ill-conditioned line.
template <typename T>
__global__ __launch_bounds__(256) void k_pois_x(Dims d, const T* __restrict__ lam_y, const T* __restrict__ lam_z,
                                                T* __restrict__ P, T* __restrict__ CC, const double* __restrict__ lam00)
{
    const long nm = (long)d.ny * d.nz;
    const long l = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= nm) return;
    const int jy = (int)(l / d.nz), kz = (int)(l % d.nz);
    if (l == 0) pois_line<double, T>(d, lam00[0], lam00[1], 0, 0, 0, P, CC);
    else pois_line<T, T>(d, lam_y[jy], lam_z[kz], jy, kz, l, P, CC);
}

// The operands of a point of component F: phi at the 7 gradient points p
// (o, o -/+ sx, o -/+ sy, o -/+ 1) and at p - s_F, the six viscosities of
// A(mu_new) in coefs' order, the component and its pg.
template <typename T>
struct CorrOps { T p0[7], p1[7], m[6], q, pg; };

template <typename T, int F>
__device__ __forceinline__ void corr_load(const Dims& d, const Visc4<T>& mu, const T* __restrict__ phi,
                                          const T* __restrict__ q, const T* __restrict__ pg, long o, CorrOps<T>& c)
{
    const long sx = d.sx, sy = d.sy;
    const long sF = F == FU ? sx : F == FV ? sy : 1;
    const long pt[7] = {0, -sx, sx, -sy, sy, -1, 1};
#pragma unroll
    for (int g = 0; g < 7; g++) {
        c.p0[g] = phi[o + pt[g]];
        c.p1[g] = phi[o + pt[g] - sF];
    }
    if (F == FU) {
        c.m[0] = mu.cell[o - sx]; c.m[1] = mu.cell[o]; c.m[2] = mu.xy[o]; c.m[3] = mu.xy[o + sy];
        c.m[4] = mu.xz[o]; c.m[5] = mu.xz[o + 1];
    } else if (F == FV) {
        c.m[0] = mu.xy[o]; c.m[1] = mu.xy[o + sx]; c.m[2] = mu.cell[o - sy]; c.m[3] = mu.cell[o];
        c.m[4] = mu.yz[o]; c.m[5] = mu.yz[o + 1];
    } else {
        c.m[0] = mu.xz[o]; c.m[1] = mu.xz[o + sx]; c.m[2] = mu.yz[o]; c.m[3] = mu.yz[o + sy];
        c.m[4] = mu.cell[o - 1]; c.m[5] = mu.cell[o];
    }
    c.q = q[o];
    c.pg = pg[o];
}

// the phi gradient of component F at gradient point g (o, o -/+ sx, ...)
template <typename T, int F>
__device__ __forceinline__ T corr_grad(const Dims& d, const CorrOps<T>& c, int g)
{
    const T h = F == FU ? T(d.dx) : F == FV ? T(d.dy) : T(d.dz);
    const double rh = F == FU ? d.rdx : F == FV ? d.rdy : d.rdz;
    return divh<T>(c.p0[g] - c.p1[g], h, rh);
}

// velo_correction's new value of the component (2144-2169)
template <typename T, int F>
__device__ __forceinline__ T corr_q(const Dims& d, const CorrOps<T>& c, T facv)
{
    return c.q - facv * corr_grad<T, F>(d, c, 0);
}

// pressure_gradient's new pg (2964-3044): pg + grad phi - fac A(mu_new) grad phi
template <typename T, int F>
__device__ __forceinline__ T corr_pg_new(const Dims& d, const Phys& ph, const CorrOps<T>& c, T fac)
{
    T gr[7];
#pragma unroll
    for (int g = 0; g < 7; g++) gr[g] = corr_grad<T, F>(d, c, g);
    T ax, bx, cx, ay, by, cy, az, bz, cz;
    coef_vals<T, F>(d, ph, 0, c.m[0], c.m[1], ax, bx, cx);
    coef_vals<T, F>(d, ph, 1, c.m[2], c.m[3], ay, by, cy);
    coef_vals<T, F>(d, ph, 2, c.m[4], c.m[5], az, bz, cz);
    const T g0 = gr[0];
    const T pxx = (ax) * gr[1] + (bx) * g0 + (cx) * gr[2];
    const T pyy = (ay) * gr[3] + (by) * g0 + (cy) * gr[4];
    const T pzz = (az) * gr[5] + (bz) * g0 + (cz) * gr[6];
    return c.pg + g0 - fac * (pyy + pxx + pzz);
}

template <typename T, int F>
__device__ __forceinline__ T corr_apply(const Dims& d, const Phys& ph, const CorrOps<T>& c, T* __restrict__ q,
                                        T* __restrict__ pg, long o, T fac, T facv)
{
    const T qn = corr_q<T, F>(d, c, facv);
    q[o] = qn;
    pg[o] = corr_pg_new<T, F>(d, ph, c, fac);
    return qn;
}

// velo_correction (2144-2169): u -= dt*alpha/Re * grad(phi) on each
// component's unknowns (so neither the inlet nor the outlet face).
template <typename T>
__global__ __launch_bounds__(256) void k_velo_corr(Dims d, Phys ph, const T* __restrict__ phi, T* __restrict__ u,
                                                   T* __restrict__ v, T* __restrict__ w,
                                                   const double* __restrict__ scal, T g, T r)
{
    const int2 bt = xcd_tile();
    const int k = bt.x * blockDim.x + threadIdx.x + 1;
    const int j = bt.y * blockDim.y + threadIdx.y + 1;
    const int i = blockIdx.z + 3;
    if (k > d.nz || j > d.ny) return;
    const long o = IX(d, i, j, k);
    const T fac = T(scal[S_DT]) * (g + r) / T(ph.Re);
    // the fused kernel's expressions (corr_q) on the operands it needs
    CorrOps<T> c;
    if (j >= 2) {
        c.p0[0] = phi[o]; c.p1[0] = phi[o - d.sy]; c.q = v[o];
        v[o] = corr_q<T, FV>(d, c, fac);
    }
    if (k >= 2) {
        c.p0[0] = phi[o]; c.p1[0] = phi[o - 1]; c.q = w[o];
        w[o] = corr_q<T, FW>(d, c, fac);
    }
    if (i >= 4) {
        c.p0[0] = phi[o]; c.p1[0] = phi[o - d.sx]; c.q = u[o];
        u[o] = corr_q<T, FU>(d, c, fac);
    }
}

// Inflow/outflow trapezoids over the interior nodes of the inlet face and
// the outlet face (2171-2210), FP64, in the reference's summation order.
// Pass 1: one block per j row sums over k (the row staged in LDS, the sum
// sequential); pass 2: one block sums the row integrals over j, forms the
// deficit (2216) and adds it to the outlet face (2219-2223).
template <typename T>
__global__ __launch_bounds__(64) void k_flux_rows(Dims d, const T* __restrict__ u, double* __restrict__ part, Bt bt)
{
    __shared__ double ri[1056], ro[1056];
    // member: blockIdx.y
    u = bt_f(bt, u, blockIdx.y);
    part += blockIdx.y * bt.np;
    const int j = 1 + blockIdx.x;
    const double hz = d.dz;
    const long bi = IX(d, 3, j, 0), bo = IX(d, d.nx + 3, j, 0);
    for (int k = threadIdx.x; k <= d.nz; k += blockDim.x) { ri[k] = (double)u[bi + k]; ro[k] = (double)u[bo + k]; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double qi = 0.0, qo = 0.0;
        for (int k = 2; k <= d.nz; k++) {
            qi += 0.5 * hz * (ri[k] + ri[k - 1]);
            qo += 0.5 * hz * (ro[k] + ro[k - 1]);
        }
        part[j] = qi;
        part[1056 + j] = qo;
    }
}

// Pass 2 and the deficit's addition to the outlet face (2216-2223) in one
// launch: block j - 1 (of ny) sums the row integrals over j in the
// reference's order, forms the deficit and adds it to row j of the outlet
// face; every block forms the same value, and block 0 also stores qin,
// qout and the deficit.
template <typename T, bool B = false>
__global__ __launch_bounds__(128) void k_flux_apply(Dims d, Phys ph0, T* __restrict__ u, double* __restrict__ scal,
                                                    const double* __restrict__ part, int rk, Bt bt)
{
    __shared__ double qk_in[1056], qk_out[1056];
    __shared__ double def;
    // member: blockIdx.y
    const int m = blockIdx.y;
    const Phys& ph = bt_phys<B>(bt, ph0, m);
    u = bt_f(bt, u, m);
    scal += m * S_SIZE;
    part += m * bt.np;
    const double hy = d.dy;
    for (int j = 1 + threadIdx.x; j <= d.ny; j += blockDim.x) { qk_in[j] = part[j]; qk_out[j] = part[1056 + j]; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double qin = 0.0, qout = 0.0;
        for (int j = 2; j <= d.ny; j++) {
            qin += 0.5 * hy * (qk_in[j - 1] + qk_in[j]);
            qout += 0.5 * hy * (qk_out[j - 1] + qk_out[j]);
        }
        const double deficit = (qin - qout) / ((ph.Y2 - ph.Y1) * (ph.Z2 - ph.Z1));
        def = deficit;
        if (blockIdx.x == 0) {
            scal[S_RK + 4 * rk + 1] = qin;
            scal[S_RK + 4 * rk + 2] = qout;
            scal[S_RK + 4 * rk + 3] = deficit;
        }
    }
    __syncthreads();
    const int j = 1 + blockIdx.x;
    const T dv = T(def);
    for (int k = 1 + threadIdx.x; k <= d.nz; k += blockDim.x) {
        const long o = IX(d, d.nx + 3, j, k);
        u[o] = u[o] + dv;
    }
}

// velo_correction (2144-2169) and pressure_gradient (2964-3044) of one
// substage in one pass: both use the same phi gradient g0 at a velocity
// point, and pg reads neither u, v nor w, so updating it here, before the
// outflow deficit and the ghost copies, gives the reference's values.
template <typename T, bool B = false>
__global__ __launch_bounds__(256) void k_corr_pg(Dims d, Phys ph0, Visc4<T> mu, const T* __restrict__ phi,
                                                 T* __restrict__ u, T* __restrict__ v, T* __restrict__ w,
                                                 T* __restrict__ pgu, T* __restrict__ pgv, T* __restrict__ pgw,
                                                 const double* __restrict__ scal0, T g, T r, int vghost, Bt bt)
{
    const int2 tl = xcd_tile();
    const int k = tl.x * blockDim.x + threadIdx.x + 1;
    const int j = tl.y * blockDim.y + threadIdx.y + 1;
    int il;
    const int m = bt_member(bt, blockIdx.z, gridDim.z, il);
    const int i = il + 3;
    if (k > d.nz || j > d.ny) return;
    const Phys& ph = bt_phys<B>(bt, ph0, m);
    const double* __restrict__ scal = scal0 + m * S_SIZE;
    // every field of member m at the same offset
    const long o = IX(d, i, j, k) + m * bt.fs;
    const T fac = T(0.5) * T(scal[S_DT]) * (g + r);
    const T facv = T(scal[S_DT]) * (g + r) / T(ph.Re);
    // the three components' operands are loaded before any update, for
    // every point (the loads the three share then issue once): a point
    // whose component is no unknown reads at most two rows, planes or
    // points below its own, inside the ghost ring or the previous plane,
    // and stores nothing
    const bool dv = j >= 2, dw = k >= 2, du = i >= 4;
    CorrOps<T> cv, cw, cu;
    corr_load<T, FV>(d, mu, phi, v, pgv, o, cv);
    corr_load<T, FW>(d, mu, phi, w, pgw, o, cw);
    corr_load<T, FU>(d, mu, phi, u, pgu, o, cu);
    // with vghost, update_veloghost_points for the values just written
    if (dv) {
        const T val = corr_apply<T, FV>(d, ph, cv, v, pgv, o, fac, facv);
        if (vghost) velo_ghost_point<T>(d, FV, v + o, i, j, k, val);
    }
    if (dw) {
        const T val = corr_apply<T, FW>(d, ph, cw, w, pgw, o, fac, facv);
        if (vghost) velo_ghost_point<T>(d, FW, w + o, i, j, k, val);
    }
    if (du) {
        const T val = corr_apply<T, FU>(d, ph, cu, u, pgu, o, fac, facv);
        if (vghost) velo_ghost_point<T>(d, FU, u + o, i, j, k, val);
    }
}

// What k_corr_pg_run holds of phi and the viscosities around a thread's KP points
// (k .. k + K - 1 of row j): names say the row (c: j, m: j - 1, p: j + 1,
// mm: j - 2), the plane (1: i + 1, none: i, b: i - 1, bb: i - 2) and the runs'
// first k.
template <typename T>
struct CorrRuns {
    static constexpr int K = KP<T>::value;
    T c[K + 3], m[K + 2], p[K + 1], mm[K];   // plane i: from k - 2, k - 1, k - 1, k
    T c1[K + 1], m1[K];                      // plane i + 1: from k - 1, k
    T cb[K + 2], mb[K], pb[K], cbb[K];       // plane i - 1: from k - 1, k, k; plane i - 2: k
    T cell[K + 1], cellm[K], cellb[K];       // mu.cell: from k - 1; row j - 1; plane i - 1
    T xy[K], xyp[K], xy1[K], xz[K + 1], xz1[K], yz[K + 1], yzp[K];

    // component F's operands of point q (corr_load's)
    template <int F>
    __device__ __forceinline__ void ops(int q, CorrOps<T>& o) const
    {
        const T x0[7] = {c[q + 2], cb[q + 1], c1[q + 1], m[q + 1], p[q + 1], c[q + 1], c[q + 3]};
        const T xu[7] = {cb[q + 1], cbb[q], c[q + 2], mb[q], pb[q], cb[q], cb[q + 2]};
        const T xv[7] = {m[q + 1], mb[q], m1[q], mm[q], c[q + 2], m[q], m[q + 2]};
        const T xw[7] = {c[q + 1], cb[q], c1[q], m[q], p[q], c[q], c[q + 2]};
#pragma unroll
        for (int g = 0; g < 7; g++) {
            o.p0[g] = x0[g];
            o.p1[g] = F == FU ? xu[g] : F == FV ? xv[g] : xw[g];
        }
        if (F == FU) {
            o.m[0] = cellb[q]; o.m[1] = cell[q + 1]; o.m[2] = xy[q]; o.m[3] = xyp[q]; o.m[4] = xz[q]; o.m[5] = xz[q + 1];
        } else if (F == FV) {
            o.m[0] = xy[q]; o.m[1] = xy1[q]; o.m[2] = cellm[q]; o.m[3] = cell[q + 1]; o.m[4] = yz[q]; o.m[5] = yz[q + 1];
        } else {
            o.m[0] = xz[q]; o.m[1] = xz1[q]; o.m[2] = yz[q]; o.m[3] = yzp[q]; o.m[4] = cell[q]; o.m[5] = cell[q + 1];
        }
    }
};

// k_corr_pg on launches of many waves: a thread takes KP points in k and
// CORR_PLANES consecutive planes, the two planes behind it, and of the plane
// ahead what it shares with the next point, in registers (26 loads a point in
// FP32 and half as many 16-byte ones in FP64 instead of 38).  us, k_corr_pg ->
// this at 1, 2, 4, 8 planes: 256x128x128 FP64 134 -> 125, 126, 124, 128, mixed
// 71 -> 71, 68, 70, 77; 512x256x256 FP64 1043 -> 985, 964, 973, 999, mixed 537
// -> 536, 517, 509, 525; 256x96x96 mixed 39 -> 38, 37, 41, 44; 150x70x51 mixed
// 12.9 -> 13.9, 12.0, 12.7, 17.7; 64x32x32 FP64 5.3 -> 6.9, 9.6, 15, 27: with
// few waves the longer chain of a thread is what counts, hence the two forms
// (correction_and_gradient).  Bound by the
// memory: 20 fields at 256x128x128 FP64, 5.6 TB/s (one plane a thread: 16.8 at 4.4).
constexpr int CORR_PLANES = 2;
template <typename T, bool B = false>
__global__ __launch_bounds__(256) void k_corr_pg_run(Dims d, Phys ph0, Visc4<T> mu, const T* __restrict__ phi,
                                                 T* __restrict__ u, T* __restrict__ v, T* __restrict__ w,
                                                 T* __restrict__ pgu, T* __restrict__ pgv, T* __restrict__ pgw,
                                                 const double* __restrict__ scal0, T g, T r, int vghost, Bt bt)
{
    constexpr int K = KP<T>::value, np = CORR_PLANES;
    const int2 tl = xcd_tile();
    const int k0 = (tl.x * blockDim.x + threadIdx.x) * K + 1;
    const int j = tl.y * blockDim.y + threadIdx.y + 1;
    int il;
    const int m = bt_member(bt, blockIdx.z, gridDim.z, il);
    int i = il * np + 3;
    const int ie = min(i + np - 1, d.nx + 2);
    if (k0 > d.nz || j > d.ny) return;
    const Phys& ph = bt_phys<B>(bt, ph0, m);
    const double* __restrict__ scal = scal0 + m * S_SIZE;
    const T fac = T(0.5) * T(scal[S_DT]) * (g + r);
    const T facv = T(scal[S_DT]) * (g + r) / T(ph.Re);
    const long sx = d.sx, sy = d.sy;
    const T *cell = mu.cell, *xy = mu.xy, *xz = mu.xz, *yz = mu.yz;
    unsigned l = (unsigned)((j * d.sy + k0) * sizeof(T));
    long o = (long)i * sx + m * bt.fs;   // every field of member m at the same offset
    // the operands of all three components are loaded for every point: a
    // point whose component is no unknown reads at most two rows, planes or
    // points below its own, inside the ghost ring or the previous plane, and
    // stores nothing
    CorrRuns<T> e;
    lane_run(phi, o - 1, l, e.c1);
    lane_run(phi, o - sy, l, e.m1);
    {
        T t[K + 2];
        lane_run(phi, o - sx - 1, l, t);
#pragma unroll
        for (int q = 0; q < K + 2; q++) e.c[q + 1] = t[q];
        T x[K], y[K], z[K];
        lane_run(phi, o - sx - sy, l, x);
        lane_run(phi, o - sx + sy, l, y);
        lane_run(phi, o - 2 * sx, l, z);
#pragma unroll
        for (int q = 0; q < K; q++) { e.m[q + 1] = x[q]; e.p[q + 1] = y[q]; e.cb[q + 1] = z[q]; }
        lane_run(cell, o - sx, l, x);
#pragma unroll
        for (int q = 0; q < K; q++) e.cell[q + 1] = x[q];
    }
    lane_run(xy, o, l, e.xy1);
    lane_run(xz, o, l, e.xz1);
#pragma unroll 1
    for (; i <= ie; i++, o += sx) {
        per_block(l, o);
#pragma unroll
        for (int q = 0; q < K; q++) {
            e.cbb[q] = e.cb[q + 1];
            e.mb[q] = e.m[q + 1];
            e.pb[q] = e.p[q + 1];
            e.cellb[q] = e.cell[q + 1];
            e.xy[q] = e.xy1[q];
            e.xz[q] = e.xz1[q];
            e.m[q + 1] = e.m1[q];
        }
#pragma unroll
        for (int q = 0; q < K + 2; q++) e.cb[q] = e.c[q + 1];
#pragma unroll
        for (int q = 0; q < K + 1; q++) e.c[q + 1] = e.c1[q];
        lane_run(phi, o + sx - 1, l, e.c1);
        lane_run(phi, o + sx - sy, l, e.m1);
        e.c[0] = lane_at(phi, o - 2, l);
        e.c[K + 2] = lane_at(phi, o + K, l);
        e.m[0] = lane_at(phi, o - sy - 1, l);
        e.m[K + 1] = lane_at(phi, o - sy + K, l);
        lane_run(phi, o + sy - 1, l, e.p);
        lane_run(phi, o - 2 * sy, l, e.mm);
        lane_run(cell, o - 1, l, e.cell);
        lane_run(cell, o - sy, l, e.cellm);
        lane_run(xy, o + sy, l, e.xyp);
        lane_run(xy, o + sx, l, e.xy1);
        e.xz[K] = lane_at(xz, o + K, l);
        lane_run(xz, o + sx, l, e.xz1);
        lane_run(yz, o, l, e.yz);
        lane_run(yz, o + sy, l, e.yzp);
        T qv[K], qw[K], qu[K], gv[K], gw[K], gu[K];
        lane_run(v, o, l, qv);
        lane_run(w, o, l, qw);
        lane_run(u, o, l, qu);
        lane_run(pgv, o, l, gv);
        lane_run(pgw, o, l, gw);
        lane_run(pgu, o, l, gu);
#pragma unroll
        for (int q = 0; q < K; q++) {
            CorrOps<T> co;
            e.template ops<FV>(q, co);
            co.q = qv[q]; co.pg = gv[q];
            qv[q] = corr_q<T, FV>(d, co, facv);
            gv[q] = corr_pg_new<T, FV>(d, ph, co, fac);
            e.template ops<FW>(q, co);
            co.q = qw[q]; co.pg = gw[q];
            qw[q] = corr_q<T, FW>(d, co, facv);
            gw[q] = corr_pg_new<T, FW>(d, ph, co, fac);
            e.template ops<FU>(q, co);
            co.q = qu[q]; co.pg = gu[q];
            qu[q] = corr_q<T, FU>(d, co, facv);
            gu[q] = corr_pg_new<T, FU>(d, ph, co, fac);
        }
        per_block(l, o);
        if (j >= 2) {
            lane_put(v, o, l, qv, k0, 1, d.nz);
            lane_put(pgv, o, l, gv, k0, 1, d.nz);
        }
        if (k0 + K > 2) {
            lane_put(w, o, l, qw, k0, 2, d.nz);
            lane_put(pgw, o, l, gw, k0, 2, d.nz);
        }
        if (i >= 4) {
            lane_put(u, o, l, qu, k0, 1, d.nz);
            lane_put(pgu, o, l, gu, k0, 1, d.nz);
        }
        // with vghost, update_veloghost_points for the values just written
        if (vghost) {
#pragma unroll
            for (int q = 0; q < K; q++) {
                const int k = k0 + q;
                if (k > d.nz) break;
                if (j >= 2) velo_ghost_point<T>(d, FV, &lane_at(v, o + q, l), i, j, k, qv[q]);
                if (k >= 2) velo_ghost_point<T>(d, FW, &lane_at(w, o + q, l), i, j, k, qw[q]);
                if (i >= 4) velo_ghost_point<T>(d, FU, &lane_at(u, o + q, l), i, j, k, qu[q]);
            }
        }
    }
}

// pressure_gradient alone (2964-3044): pg += grad(phi) - fac A(mu_new)
// grad(phi) for the components in mask (bit 0 u, 1 v, 2 w) at their
// unknowns; the gradients at the 7 stencil points are recomputed from phi.
template <typename T>
__global__ __launch_bounds__(256) void k_pg(Dims d, Phys ph, Visc4<T> mu, const T* __restrict__ phi,
                                            T* __restrict__ pgu, T* __restrict__ pgv, T* __restrict__ pgw,
                                            const double* __restrict__ scal, T g, T r, int mask)
{
    const int2 bt = xcd_tile();
    const int k = bt.x * blockDim.x + threadIdx.x + 1;
    const int j = bt.y * blockDim.y + threadIdx.y + 1;
    const int i = blockIdx.z + 3;
    if (k > d.nz || j > d.ny) return;
    const T fac = T(0.5) * T(scal[S_DT]) * (g + r);
    const long o = IX(d, i, j, k);
    // the fused kernel's expressions (corr_pg_new); q is not used
    CorrOps<T> c;
    if ((mask & 2) && j >= 2) { corr_load<T, FV>(d, mu, phi, pgv, pgv, o, c); pgv[o] = corr_pg_new<T, FV>(d, ph, c, fac); }
    if ((mask & 1) && i >= 4) { corr_load<T, FU>(d, mu, phi, pgu, pgu, o, c); pgu[o] = corr_pg_new<T, FU>(d, ph, c, fac); }
    if ((mask & 4) && k >= 2) { corr_load<T, FW>(d, mu, phi, pgw, pgw, o, c); pgw[o] = corr_pg_new<T, FW>(d, ph, c, fac); }
}

// ------------------------------------------------------------ reductions

// find_cfl (3095-3118), pass 1: per-block max of
// |u|/dx + |v|/dy + |w|/dz at cell centres.  A block covers its tile of (j, k)
// in CFL_PLANES planes, all their loads in flight together; the max within
// a wave by lane exchange, over the waves through LDS (a max in any order is
// the same value).
constexpr int CFL_PLANES = 4;
template <typename T>
__global__ __launch_bounds__(256) void k_cfl_partial(Dims d, const T* __restrict__ u, const T* __restrict__ v,
                                                     const T* __restrict__ w, double* __restrict__ part, Bt bt)
{
    __shared__ double red[4];
    const int2 tl = xcd_tile();
    const int k = tl.x * blockDim.x + threadIdx.x + 1;
    const int j = tl.y * blockDim.y + threadIdx.y + 1;
    int ib;
    const int mb = bt_member(bt, blockIdx.z, gridDim.z, ib);
    const int t = threadIdx.y * blockDim.x + threadIdx.x;
    double m = 0.0;
    if (k <= d.nz && j <= d.ny) {
        const long o = IX(d, ib * CFL_PLANES + 3, j, k) + mb * bt.fs;
        const int n = min(CFL_PLANES, d.nx - ib * CFL_PLANES);
        T u0[CFL_PLANES + 1], v0[CFL_PLANES], v1[CFL_PLANES], w0[CFL_PLANES], w1[CFL_PLANES];
        u0[0] = u[o];
#pragma unroll
        for (int p = 0; p < CFL_PLANES; p++) {
            const long q = o + (long)min(p, n - 1) * d.sx;   // the last plane again past the end
            u0[p + 1] = u[q + d.sx];
            v0[p] = v[q];
            v1[p] = v[q + d.sy];
            w0[p] = w[q];
            w1[p] = w[q + 1];
        }
#pragma unroll
        for (int p = 0; p < CFL_PLANES; p++) {
            if (p < n) {
                const double uv = 0.5 * ((double)u0[p] + (double)u0[p + 1]);
                const double vv = 0.5 * ((double)v0[p] + (double)v1[p]);
                const double wv = 0.5 * ((double)w0[p] + (double)w1[p]);
                const double x = (fabs(uv) / d.dx) + (fabs(vv) / d.dy) + (fabs(wv) / d.dz);
                m = m > x ? m : x;
            }
        }
    }
    // the last wave of a tile may have fewer than 64 lanes
    const int lane = t & 63, nl = min(64, (int)(blockDim.x * blockDim.y) - (t - lane));
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const double x = __shfl_xor(m, s);
        m = (lane ^ s) < nl && x > m ? x : m;
    }
    if (lane == 0) red[t >> 6] = m;
    __syncthreads();
    if (t == 0) {
        const int nw = (blockDim.x * blockDim.y + 63) >> 6;
        for (int s = 1; s < nw; s++) m = m > red[s] ? m : red[s];
        part[mb * bt.np + ((long)ib * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = m;
    }
}

// bulk_velo (3381-3398): the signed u of largest |u| on the plane iend,
// the first hit in (j,k) order winning ties.  Pass 1: per-block candidates
// (value, scan index); pass 2: one block picks the winner, and advances the
// device copy of tval by (gamma+rho)*dt (pllcart3d.c:166).
__device__ __forceinline__ bool bulk_better(double b, long ib, double a, long ia)
{
    if (ib < 0) return false;
    if (ia < 0) return true;
    if (fabs(b) > fabs(a)) return true;
    if (fabs(b) < fabs(a)) return false;
    return ib < ia;
}

template <typename T>
__global__ __launch_bounds__(256) void k_bulk_partial(Dims d, const T* __restrict__ u, double* __restrict__ part)
{
    __shared__ double sv[256];
    __shared__ long si[256];
    const int t = threadIdx.x;
    const int np = d.ny * d.nz;
    const int l = blockIdx.x * blockDim.x + t;
    double v = 0.0;
    long id = -1;
    if (l < np) {
        const double x = (double)u[IX(d, d.nx + 2, 1 + l / d.nz, 1 + l % d.nz)];
        if (fabs(x) > 0.0) { v = x; id = l; }
    }
    sv[t] = v; si[t] = id;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s && bulk_better(sv[t + s], si[t + s], sv[t], si[t])) { sv[t] = sv[t + s]; si[t] = si[t + s]; }
        __syncthreads();
    }
    if (t == 0) { part[2 * blockIdx.x] = sv[0]; part[2 * blockIdx.x + 1] = (double)si[0]; }
}

template <typename T>
__global__ __launch_bounds__(256) void k_bulk_final(const double* __restrict__ part, int nb, double* __restrict__ scal,
                                                    int rk, double alpha, double* __restrict__ tval)
{
    __shared__ double sv[256];
    __shared__ long si[256];
    const int t = threadIdx.x;
    double v = 0.0;
    long id = -1;
    for (int b = t; b < nb; b += blockDim.x) {
        const double x = part[2 * b];
        const long ix = (long)part[2 * b + 1];
        if (bulk_better(x, ix, v, id)) { v = x; id = ix; }
    }
    sv[t] = v; si[t] = id;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s && bulk_better(sv[t + s], si[t + s], sv[t], si[t])) { sv[t] = sv[t + s]; si[t] = si[t + s]; }
        __syncthreads();
    }
    if (t == 0) {
        scal[S_RK + 4 * rk] = si[0] < 0 ? 0.0 : sv[0];
        if (tval) tval[0] = tval[0] + alpha * scal[S_DT];
    }
}

// bulk_velo in one block of BULK_NT threads over the whole plane (ny nz <=
// BULK1_MAX): each thread scans its points in increasing index, then a tree
// over the block; the winner (largest |u|, first index among ties) is the
// same in any order.
constexpr int BULK1_MAX = 65536, BULK_NT = 1024;
template <typename T>
__device__ __forceinline__ void bulk_block(const Dims& d, const T* u, double* __restrict__ out, double* sv, long* si)
{
    constexpr int NT = BULK_NT, U = 8;
    const int t = threadIdx.x;
    const int np = d.ny * d.nz;
    const T* pl = u + IX(d, d.nx + 2, 1, 1);
    double v = 0.0;
    long id = -1;
    auto take = [&](double x, long l) {
        if (fabs(x) > 0.0 && bulk_better(x, l, v, id)) { v = x; id = l; }
    };
    int l = t;
    for (; l + (U - 1) * NT < np; l += U * NT) {
        T x[U];
#pragma unroll
        for (int q = 0; q < U; q++) {
            const int m = l + q * NT;
            x[q] = pl[(long)(m / d.nz) * d.sy + m % d.nz];
        }
#pragma unroll
        for (int q = 0; q < U; q++) take((double)x[q], l + q * NT);
    }
    for (; l < np; l += NT) take((double)pl[(long)(l / d.nz) * d.sy + l % d.nz], l);
    sv[t] = v; si[t] = id;
    __syncthreads();
    for (int s2 = NT / 2; s2 > 0; s2 >>= 1) {
        if (t < s2 && bulk_better(sv[t + s2], si[t + s2], sv[t], si[t])) { sv[t] = sv[t + s2]; si[t] = si[t + s2]; }
        __syncthreads();
    }
    if (t == 0) *out = si[0] < 0 ? 0.0 : sv[0];
}

// pass 2: max over the partials; dt = min(CFLmax/max, Timestep)
// (pllcart3d.c:159-160, 3115)
// (one block of 1024 threads, eight loads per thread in flight per round;
// a max in any order is the same value).  With tval the first substage's start
// rides in the launch: block row 1 computes bulk_velo's value, row 2 the stale
// values, and row 0 advances tval by alpha dt.
template <typename T>
__global__ __launch_bounds__(1024) void k_cfl_final(const double* __restrict__ part, long np, double CFLmax,
                                                    double Timestep, double* __restrict__ scal, Dims d, double alpha,
                                                    double* __restrict__ tval, const T* __restrict__ q0,
                                                    const T* __restrict__ q1, const T* __restrict__ q2,
                                                    const T* __restrict__ q3, T* __restrict__ stale, Bt bt)
{
    constexpr int NT = 1024, U = 8;
    static_assert(NT == BULK_NT, "a bulk_block");
    __shared__ double red[NT];
    __shared__ long si[NT];
    if (blockIdx.y) {
        const int m = blockIdx.x;
        if (blockIdx.y == 1)
            bulk_block<T>(d, bt_f(bt, q1, m), scal + m * S_SIZE + S_RK, red, si);
        else if (threadIdx.x < 16)
            stale[m * 16 + threadIdx.x] = stale_value<T>(d, bt_f(bt, q0, m), bt_f(bt, q1, m), bt_f(bt, q2, m),
                                                         bt_f(bt, q3, m), threadIdx.x);
        return;
    }
    // member: blockIdx.x
    if (bt.ph) {
        CFLmax = bt.ph[blockIdx.x].CFLmax;
        Timestep = bt.ph[blockIdx.x].Timestep;
    }
    part += blockIdx.x * bt.np;
    scal += blockIdx.x * S_SIZE;
    const int t = threadIdx.x;
    double m = 0.0;
    long l = t;
    for (; l + (U - 1) * NT < np; l += U * NT) {
        double a[U];
#pragma unroll
        for (int q = 0; q < U; q++) a[q] = part[l + q * NT];
#pragma unroll
        for (int q = 0; q < U; q++) m = m > a[q] ? m : a[q];
    }
    for (; l < np; l += NT) m = m > part[l] ? m : part[l];
    red[t] = m;
    __syncthreads();
    for (int s = NT / 2; s > 0; s >>= 1) {
        if (t < s) red[t] = red[t] > red[t + s] ? red[t] : red[t + s];
        __syncthreads();
    }
    if (t == 0) {
        const double cfldt = CFLmax / red[0];
        scal[S_CFL] = red[0];
        const double dt = (cfldt < Timestep) ? cfldt : Timestep;
        scal[S_DT] = dt;
        if (tval) tval[blockIdx.x] = tval[blockIdx.x] + alpha * dt;
    }
}

// bulk_velo, and with q0 set the 16 stale values (k_stale) in block 1
template <typename T>
__global__ __launch_bounds__(1024) void k_bulk_stale(Dims d, const T* __restrict__ u, double* __restrict__ scal,
                                                     int rk, double alpha, double* __restrict__ tval,
                                                     const T* __restrict__ q0, const T* __restrict__ q1,
                                                     const T* __restrict__ q2, const T* __restrict__ q3,
                                                     T* __restrict__ stale, Bt bt)
{
    __shared__ double sv[BULK_NT];
    __shared__ long si[BULK_NT];
    // member: blockIdx.y
    const int mb = blockIdx.y, t = threadIdx.x;
    scal += mb * S_SIZE;
    if (blockIdx.x == 1) {
        if (t < 16)
            stale[mb * 16 + t] = stale_value<T>(d, bt_f(bt, q0, mb), bt_f(bt, q1, mb), bt_f(bt, q2, mb),
                                                bt_f(bt, q3, mb), t);
        return;
    }
    bulk_block<T>(d, bt_f(bt, u, mb), scal + S_RK + 4 * rk, sv, si);
    if (t == 0 && tval) tval[mb] = tval[mb] + alpha * scal[S_DT];
}

// What a substage ends with on planes of at most FE_MAX x FE_MAX, and what
// the next one starts with, in one launch instead of three (k_flux_rows,
// k_flux_apply, k_bulk_stale: 4.7 to 5.4 us each at 64x32x32, the floor of a
// launch): block 0 sums both faces' rows as k_flux_rows does (FE_K columns of
// every row at a time through LDS, the next ones in flight; a thread a row),
// forms and adds the deficit as k_flux_apply does, and with next >= 0
// computes the 16 stale values (they may read the outlet face) of the new
// fields; block 1 then computes bulk_velo's value for substage next (its plane
// is the one before the outlet face) and advances tval.  us, the three launches
// -> this: 64x32x32 FP64 14 -> 5.4, 150x70x51 mixed 15 -> 8.2, 256x128x128 FP64
// 22 -> 19, mixed 21 -> 15; the sums' serial chains are what is left, so larger
// planes keep a block per row.
constexpr int FE_MAX = 128, FE_K = 16;
template <typename T, bool B = false>
__global__ __launch_bounds__(1024) void k_step_end(Dims d, Phys ph0, T* u0, double* __restrict__ scal, int rk, int next,
                                                   double alpha, double* __restrict__ tval, const T* __restrict__ q0,
                                                   const T* __restrict__ q2, const T* __restrict__ q3,
                                                   T* __restrict__ stale, Bt bt)
{
    __shared__ union {
        struct { double x[2][FE_MAX][FE_K + 1], rows[2][FE_MAX + 1], sum[2]; } f;
        struct { double sv[BULK_NT]; long si[BULK_NT]; } b;
    } sh;
    // member: blockIdx.y
    const int m = blockIdx.y, t = threadIdx.x;
    T* u = bt_f(bt, u0, m);
    scal += m * S_SIZE;
    if (blockIdx.x == 1) {
        bulk_block<T>(d, u, scal + S_RK + 4 * next, sh.b.sv, sh.b.si);
        if (t == 0) tval[m] = tval[m] + alpha * scal[S_DT];
        return;
    }
    const Phys& ph = bt_phys<B>(bt, ph0, m);
    const T* face[2] = {u + IX(d, 3, 1, 1), u + IX(d, d.nx + 3, 1, 1)};
    constexpr int U = 2 * FE_MAX * FE_K / 1024;
    T v[U];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int q = 0; q < U; q++) {
            const int e = t + 1024 * q, k = k0 + (e & (FE_K - 1)), r = (e / FE_K) & (FE_MAX - 1), s = e / (FE_K * FE_MAX);
            if (r < d.ny && k < d.nz) v[q] = face[s][(long)r * d.sy + k];
        }
    };
    const int s = t >> 7, r = t & (FE_MAX - 1);   // the face and row of t < 256
    const bool sums = t < 2 * FE_MAX && r < d.ny;
    const double hz = d.dz, hy = d.dy;
    double q = 0.0, last = 0.0;
    fetch(0);
    for (int k0 = 0; k0 < d.nz; k0 += FE_K) {
        __syncthreads();   // the columns before read
#pragma unroll
        for (int p = 0; p < U; p++) {
            const int e = t + 1024 * p;
            sh.f.x[e / (FE_K * FE_MAX)][(e / FE_K) & (FE_MAX - 1)][e & (FE_K - 1)] = (double)v[p];
        }
        __syncthreads();
        if (k0 + FE_K < d.nz) fetch(k0 + FE_K);
        if (sums) {
            const int n = min(FE_K, d.nz - k0);
            for (int k = 0; k < n; k++) {
                const double x = sh.f.x[s][r][k];
                if (k0 + k > 0) q += 0.5 * hz * (x + last);
                last = x;
            }
        }
    }
    if (sums) sh.f.rows[s][r + 1] = q;
    __syncthreads();
    if (t == 0 || t == 64) {   // a wave each
        const double* qk = sh.f.rows[t >> 6];
        double a = 0.0;
        for (int j = 2; j <= d.ny; j++) a += 0.5 * hy * (qk[j - 1] + qk[j]);
        sh.f.sum[t >> 6] = a;
    }
    __syncthreads();
    const double qin = sh.f.sum[0], qout = sh.f.sum[1];
    const double deficit = (qin - qout) / ((ph.Y2 - ph.Y1) * (ph.Z2 - ph.Z1));
    if (t == 0) {
        scal[S_RK + 4 * rk + 1] = qin;
        scal[S_RK + 4 * rk + 2] = qout;
        scal[S_RK + 4 * rk + 3] = deficit;
    }
    const T dv = T(deficit);
    T* out = u + IX(d, d.nx + 3, 1, 1);
    for (int e = t; e < d.ny * FE_MAX; e += 1024) {
        const int j = e / FE_MAX, k = e & (FE_MAX - 1);
        if (k < d.nz) out[(long)j * d.sy + k] += dv;
    }
    if (next < 0) return;
    __syncthreads();
    if (t < 16) stale[m * 16 + t] = stale_value<T>(d, bt_f(bt, q0, m), u, bt_f(bt, q2, m), bt_f(bt, q3, m), t);
}

// ---------------------------------------------------------------- DCT GEMM

// Dense DCT contractions (fftw_3d.h REDFT10 / REDFT01 as matrices) on the
// matrix cores:
//   TRB = true : C[b] (M x N) = A[b] (M x K) * B^T, B stored N x K
//   TRB = false: C[b] (M x N) = A[b] (M x K) * B[b], B stored K x N
// One 16x16x4 MFMA per step (V_MFMA_F64_16X16X4_F64 / V_MFMA_F32_16X16X4_F32):
// lane l supplies A[l%16][k0 + l/16] and B[k0 + l/16][l%16]; its four
// results are C[row][l%16] with row = l/16 + 4r for FP64 and 4(l/16) + r for
// FP32, r = 0..3 (both measured on gfx950 with single-lane probes).  Block
// tile 64 x 128 (4 wavefronts of 32 x 64, 2 x 4 MFMA tiles each), K chunks of
// 16 double-buffered in LDS.  Every output accumulates over k in increasing
// order with fused multiply-adds; FFTW's fast transforms round differently
// from any direct sum, so the results agree with the reference's REDFT10/01
// to rounding.
template <typename T> struct Mma;
template <> struct Mma<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ int row(int lk, int r) { return lk + 4 * r; }
    static __device__ __forceinline__ acc run(double a, double b, acc c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};
template <> struct Mma<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
    static __device__ __forceinline__ acc run(float a, float b, acc c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};

// Source of a forward transform's first contraction: the packed block `in`, or
// with u set the Poisson right-hand side itself, Re / (dt (g + r)) times the
// divergence of the new velocities (k_div's expressions), so that the packed
// block is not made first (one launch and two passes over it less).  us, k_div
// and the transform -> this: 256x128x128 FP64 58 -> 46, mixed 39 -> 27;
// 512x256x256 FP64 395 -> 344, mixed 190 -> 121 (rows pass); 256x96x96 mixed 31
// -> 25; 64x32x32 FP64 10 -> 6.8.
template <typename T>
struct DivIn {
    const T *u, *v, *w;
    const double* scal;
    Dims d;
    double Re;
    T gr;
    // member m's factor
    __device__ __forceinline__ T fac(const Bt& bt, int m) const
    {
        const double re = bt.ph ? bt.ph[m].Re : Re;
        return T(re) / (T(scal[m * S_SIZE + S_DT]) * gr);
    }
    // point (x, y, z) of the packed block, from the member's first value on
    __device__ __forceinline__ T at(long mo, T fac, int x, int y, int z) const
    {
        const long o = IX(d, x + 3, y + 1, z + 1) + mo;
        const T dvx = divh<T>(u[o + d.sx] - u[o], T(d.dx), d.rdx);
        const T dvy = divh<T>(v[o + d.sy] - v[o], T(d.dy), d.rdy);
        const T dvz = divh<T>(w[o + 1] - w[o], T(d.dz), d.rdz);
        const T dv = (dvx + dvy + dvz);
        return fac * dv;
    }
};

// Epilogue of the last inverse contraction when phi is set: batch b, row
// gm, column gn of the packed [x][y][z] block is phi's interior point
// (3 + b, 1 + gm, 1 + gn), divided by the inverse transform's norm 4 ny nz
// (fftw_3d.h:101); with ghosts, a point next to a face also writes its
// face ghost copy (update_phi_ghosts, 2758-2807).
template <typename T>
struct PhiOut { T* phi; long sx, sy; int nx, ny, nz, ghosts; };

// phi's interior point (3 + b, 1 + gm, 1 + gn) from the inverse transform's
// value val (already normalised), and with ghosts its face ghost copies
template <typename T>
__device__ __forceinline__ void phi_store(const PhiOut<T>& po, int b, int gm, int gn, T val)
{
    const long o = (long)(3 + b) * po.sx + (long)(1 + gm) * po.sy + (1 + gn);
    po.phi[o] = val;
    if (po.ghosts) {
        if (gn == 0) po.phi[o - 1] = val;
        if (gn == po.nz - 1) po.phi[o + 1] = val;
        if (gm == 0) po.phi[o - po.sy] = val;
        if (gm == po.ny - 1) po.phi[o + po.sy] = val;
        if (b == 0) po.phi[o - po.sx] = val;
        if (b == po.nx - 1) po.phi[o + po.sx] = val;
    }
}

#ifndef GEMM_BK
#define GEMM_BK 16
#endif

template <typename T, bool TRB>
__global__ __launch_bounds__(256) void k_gemm(int M, int N, int K, const T* __restrict__ A, long sA,
                                              const T* __restrict__ B, long sB, T* __restrict__ C, long sC,
                                              PhiOut<T> po)
{
    constexpr int BM = 64, BN = 128, BK = GEMM_BK;
    constexpr int NA = BM * BK / 256, NB = BN * BK / 256;   // per-thread loads per chunk
    // two LDS buffers: the next chunk's global loads are in flight (in
    // registers) while the matrix cores work on the current one
    __shared__ T As[2][BK][BM + 1];
    __shared__ T Bs[2][BK][BN + 1];
    typedef typename Mma<T>::acc acc_t;
    const int b = blockIdx.z;
    A += (long)b * sA; B += (long)b * sB; C += (long)b * sC;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 64;
    const int li = lane & 15, lk = lane >> 4;
    acc_t acc[2][4];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int t = 0; t < 4; t++) acc[s][t] = acc_t{T(0), T(0), T(0), T(0)};
    T ra[NA], rb[NB];
    auto load = [&](int k0) {
#pragma unroll
        for (int p = 0; p < NA; p++) {
            const int e = threadIdx.x + 256 * p;
            const int mm = e / BK, kk = e % BK;
            const int gm = m0 + mm, gk = k0 + kk;
            ra[p] = (gm < M && gk < K) ? A[(long)gm * K + gk] : T(0);
        }
#pragma unroll
        for (int p = 0; p < NB; p++) {
            const int e = threadIdx.x + 256 * p;
            const int nn = TRB ? (e / BK) : (e % BN);
            const int kb = TRB ? (e % BK) : (e / BN);
            const int gn = n0 + nn, gkb = k0 + kb;
            T bv = T(0);
            if (gn < N && gkb < K) bv = TRB ? B[(long)gn * K + gkb] : B[(long)gkb * N + gn];
            rb[p] = bv;
        }
    };
    load(0);
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
        for (int p = 0; p < NA; p++) {
            const int e = threadIdx.x + 256 * p;
            As[buf][e % BK][e / BK] = ra[p];
        }
#pragma unroll
        for (int p = 0; p < NB; p++) {
            const int e = threadIdx.x + 256 * p;
            const int nn = TRB ? (e / BK) : (e % BN);
            const int kb = TRB ? (e % BK) : (e / BN);
            Bs[buf][kb][nn] = rb[p];
        }
        __syncthreads();
        if (k0 + BK < K) load(k0 + BK);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            T av[2], bv[4];
#pragma unroll
            for (int s = 0; s < 2; s++) av[s] = As[buf][kk + lk][wm + 16 * s + li];
#pragma unroll
            for (int t = 0; t < 4; t++) bv[t] = Bs[buf][kk + lk][wn + 16 * t + li];
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int t = 0; t < 4; t++) acc[s][t] = Mma<T>::run(av[s], bv[t], acc[s][t]);
        }
        buf ^= 1;
    }
    if (po.phi) {
        const T norm = T(4 * po.ny * po.nz);
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int gn = n0 + wn + 16 * t + li;
                if (gn >= N) continue;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int gm = m0 + wm + 16 * s + Mma<T>::row(lk, r);
                    if (gm >= M) continue;
                    phi_store(po, b, gm, gn, fdiv<T>(acc[s][t][r], norm));
                }
            }
        return;
    }
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int gn = n0 + wn + 16 * t + li;
            if (gn >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int gm = m0 + wm + 16 * s + Mma<T>::row(lk, r);
                if (gm < M) C[(long)gm * N + gn] = acc[s][t][r];
            }
        }
}

// Dense (y, z) transforms of small planes (ny and nz multiples of 16, at
// most 64: the coarse and ensemble grids), both contractions per launch.
constexpr int DS_MAX = 64;
// LDS pitch of a plane's rows: nz + 4 values (the 16 x 4 lanes of an A
// operand read rows li at column lk: li (nz + 4) + lk falls in distinct
// banks, nz + 4 being 4 times an odd number)
__host__ __device__ constexpr int ds_pitch(int nz) { return nz + 4; }

// Persistent blocks take the planes in turn (plane p of the packed blocks
// is member p / nx's plane p % nx when batched, Bt), the DCT matrices
// staged in LDS once; each plane is staged in LDS and contracted along z
// into Q[y][kz] = sum_m P[y][m] Cz[kz][m], then along y into out[ky][kz] =
// sum_m Cy[ky][m] Q[m][kz] (with phi set: phi, normalised, with its face
// ghosts).  A block's next plane is loaded into registers while it
// contracts the current one, and written to LDS once the z contraction has
// read the current one, so HBM latency overlaps the matrix work.  N > 0:
// square planes ny = nz = N (so Cy = Cz, one table staged), N / 16 waves,
// wave w making the 16 x 16 tiles of row tile w (their A operand shared),
// the k loops unrolled; N = 0: any ny, nz, 4 waves, wave w making tiles
// w, w + 4, ...  A wave's tiles' accumulators are interleaved over k.  Each
// tile's MFMA sequence is k_gemm's (a zero accumulator, k ascending in
// steps of 4), so the result equals the two k_gemm launches bit for bit,
// without Q's round trip through HBM.  A plane is read whole before any of
// it is written, by its one block: the transform is in place (io).
__host__ __device__ constexpr int dct_planes_threads(int N) { return N ? 4 * N : 256; }

template <typename T, bool INV, int N>
__global__ __launch_bounds__(256) void k_dct_planes(int ny_, int nz_, int nx, int nplanes, T* __restrict__ io,
                                                    const T* __restrict__ Cz, const T* __restrict__ Cy, PhiOut<T> po,
                                                    DivIn<T> dv, Bt bt)
{
    static_assert(N % 16 == 0 && N <= DS_MAX, "square planes of 16 .. 64");
    extern __shared__ unsigned char pllc_smem[];
    typedef typename Mma<T>::acc acc_t;
    constexpr int NT = dct_planes_threads(N);
    constexpr int TW = N ? N / 16 : (DS_MAX / 16) * (DS_MAX / 16) / 4;   // tiles per wave at most
    constexpr int PF = (N ? N * N : DS_MAX * DS_MAX) / NT;              // plane values per thread at most
    constexpr int KN = N ? N : DS_MAX;
    const int ny = N ? N : ny_, nz = N ? N : nz_;
    const int pz = ds_pitch(nz), py = ds_pitch(ny);
    T* P = reinterpret_cast<T*>(pllc_smem);   // [ny][pz]
    T* Q = P + ny * pz;                        // [ny][pz]
    T* Z = Q + ny * pz;                        // Cz [nz][pz]
    T* Y = N ? Z : Z + nz * pz;                // Cy [ny][py] (square planes: Cy = Cz)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int tz = nz >> 4, nt = (ny >> 4) * tz;
    const int plane = ny * nz;
    const T norm = T(4 * po.ny * po.nz);
    const int G = gridDim.x;
    // this wave's tiles: origin (y0, z0) and whether the tile exists
    int ty0[TW], tz0[TW];
    bool tok[TW];
#pragma unroll
    for (int u = 0; u < TW; u++) {
        if (N) { ty0[u] = 16 * wave; tz0[u] = 16 * u; tok[u] = true; }
        else {
            const int t = wave + 4 * u;
            tok[u] = t < nt;
            ty0[u] = (t / tz) * 16;
            tz0[u] = (t % tz) * 16;
        }
    }
    T pf[PF];
    auto fetch = [&](int p) {
        if (!INV && dv.u) {
            const int m = p / nx, x = p - m * nx;
            const T f = dv.fac(bt, m);
#pragma unroll
            for (int u = 0; u < PF; u++) {
                const int e = threadIdx.x + NT * u, y = e / nz;
                if (N || e < plane) pf[u] = dv.at(m * bt.fs, f, x, y, e - y * nz);
            }
            return;
        }
        const T* src = io + (long)p * plane;
#pragma unroll
        for (int u = 0; u < PF; u++) {
            const int e = threadIdx.x + NT * u;
            if (N || e < plane) pf[u] = src[e];
        }
    };
    auto put = [&]() {
#pragma unroll
        for (int u = 0; u < PF; u++) {
            const int e = threadIdx.x + NT * u;
            if (N || e < plane) {
                const int y = e / nz;
                P[y * pz + e - y * nz] = pf[u];
            }
        }
    };
    int p = blockIdx.x;
    if (p < nplanes) fetch(p);
    for (int e = threadIdx.x; e < nz * nz; e += NT) {
        const int r = e / nz;
        Z[r * pz + e - r * nz] = Cz[e];
    }
    if (!N)
        for (int e = threadIdx.x; e < ny * ny; e += NT) {
            const int r = e / ny;
            Y[r * py + e - r * ny] = Cy[e];
        }
    if (p < nplanes) put();
    if (p + G < nplanes) fetch(p + G);
    __syncthreads();
    for (; p < nplanes; p += G) {
        // P holds plane p; pf holds plane p + G (in flight)
        acc_t acc[TW];
#pragma unroll
        for (int u = 0; u < TW; u++) acc[u] = acc_t{T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int k = 0; k < KN; k += 4) {
            if (N || k < nz) {
#pragma unroll
                for (int u = 0; u < TW; u++)
                    if (tok[u])
                        acc[u] = Mma<T>::run(P[(ty0[u] + li) * pz + k + lk], Z[(tz0[u] + li) * pz + k + lk], acc[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < TW; u++)
            if (tok[u]) {
#pragma unroll
                for (int r = 0; r < 4; r++) Q[(ty0[u] + Mma<T>::row(lk, r)) * pz + tz0[u] + li] = acc[u][r];
            }
        __syncthreads();   // P read by every wave, Q written
        if (p + G < nplanes) put();
        if (p + 2 * G < nplanes) fetch(p + 2 * G);
#pragma unroll
        for (int u = 0; u < TW; u++) acc[u] = acc_t{T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int k = 0; k < KN; k += 4) {
            if (N || k < ny) {
#pragma unroll
                for (int u = 0; u < TW; u++)
                    if (tok[u])
                        acc[u] = Mma<T>::run(Y[(ty0[u] + li) * py + k + lk], Q[(k + lk) * pz + tz0[u] + li], acc[u]);
            }
        }
        const int m = p / nx, x = p - m * nx;
        PhiOut<T> pm = po;
        pm.phi = bt_f(bt, po.phi, m);
#pragma unroll
        for (int u = 0; u < TW; u++) {
            if (!tok[u]) continue;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int gm = ty0[u] + Mma<T>::row(lk, r), gn = tz0[u] + li;
                if (INV && po.phi) phi_store(pm, x, gm, gn, fdiv<T>(acc[u][r], norm));
                else io[(long)p * plane + (long)gm * nz + gn] = acc[u][r];
            }
        }
        __syncthreads();   // Q read by every wave, P holds plane p + G
    }
}

// Dense (y, z) transforms of any plane up to DW_MAX x DW_MAX, both contractions
// in one launch: one block per plane, which lies in LDS padded with zeros to
// whole 16 x 16 tiles; the z contraction's tiles are held in registers until
// every wave has read the plane and then take its place.  A wave makes R
// tiles that share one operand of the DCT matrix, which it reads from the
// matrix laid out in operand order (O[(tile row, k / 4)][lane], zero-padded:
// one coalesced load per matrix instruction group, the same for every block,
// from L2), the next four steps' loads in flight.  R is the smallest that
// fits 16 waves (dw_share).  The MFMA sequence of every tile is k_gemm's, so
// the result equals the two k_gemm launches bit for bit.  us, the two k_gemm
// launches -> this, forward / inverse: 256x96x96 mixed 36 / 36 -> 19 / 21,
// 150x70x51 mixed 23 / 23 -> 11 / 12, 97x45x39 FP64 20 / 20 -> 8.4 / 9.0,
// 256x112x112 FP64 60 / 60 -> 46 / 49, 300x33x120 mixed 24 / 24 -> 24 / 25.
// k_gemm's 64 x 128 tiles were padding or too few blocks there and Q made a
// round trip; here a plane's load, its two contractions (6 us of matrix
// instructions at 96 x 96 FP32) and its store follow each other in the one
// block of a CU.  The whole plane's loads in flight at once instead of four a
// thread: no faster.  A plane is read whole before any of it is written: the
// transform is in place (io).
constexpr int DW_MAX = 128;
__host__ __device__ constexpr int dw_tiles(int n) { return (n + 15) / 16; }
__host__ __device__ constexpr int dw_pitch(int nz) { return 16 * dw_tiles(nz) + 4; }
// tiles per wave along one direction (t tiles) with `other` tiles across
__host__ __device__ constexpr int dw_share(int t, int other)
{
    int r = 1;
    while (other * ((t + r - 1) / r) > 16) r++;
    return r;
}
__host__ __device__ constexpr int dw_waves(int ny, int nz)
{
    const int ty = dw_tiles(ny), tz = dw_tiles(nz), ry = dw_share(ty, tz), rz = dw_share(tz, ty);
    const int a = tz * ((ty + ry - 1) / ry), b = ty * ((tz + rz - 1) / rz);
    return a > b ? a : b;
}

// R accumulators over kt steps of 4: op(u, k) the shared-memory operand of
// tile u, O the other one; TA: O is the A operand
template <typename T, int R, bool TA, typename F>
__device__ __forceinline__ void dw_contract(typename Mma<T>::acc (&acc)[4], const T* __restrict__ O, int kt, F op)
{
    typedef typename Mma<T>::acc acc_t;
#pragma unroll
    for (int u = 0; u < R; u++) acc[u] = acc_t{T(0), T(0), T(0), T(0)};
    T nx[4];
#pragma unroll
    for (int t = 0; t < 4; t++) nx[t] = O[64 * t];
    for (int k = 0; k < kt; k += 4) {   // kt is a multiple of 4
        T cu[4];
#pragma unroll
        for (int t = 0; t < 4; t++) cu[t] = nx[t];
        if (k + 4 < kt) {
#pragma unroll
            for (int t = 0; t < 4; t++) nx[t] = O[64 * (k + 4 + t)];
        }
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int u = 0; u < R; u++) {
                const T x = op(u, 4 * (k + t));
                acc[u] = TA ? Mma<T>::run(cu[t], x, acc[u]) : Mma<T>::run(x, cu[t], acc[u]);
            }
    }
}

template <typename T, bool INV>
__global__ __launch_bounds__(1024) void k_dct_wide(int ny, int nz, T* __restrict__ io, const T* __restrict__ Oz,
                                                   const T* __restrict__ Oy, PhiOut<T> po, DivIn<T> dv)
{
    extern __shared__ unsigned char pllc_smem[];
    typedef typename Mma<T>::acc acc_t;
    T* P = reinterpret_cast<T*>(pllc_smem);   // [16 ty][pz]
    const int ty = dw_tiles(ny), tz = dw_tiles(nz), pz = dw_pitch(nz);
    const int ry = dw_share(ty, tz), rz = dw_share(tz, ty);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const long plane = (long)ny * nz;
    const T* src = io + blockIdx.x * plane;
    const int cells = 256 * ty * tz, nzp = 16 * tz;
    const bool fused = !INV && dv.u;
    const T f = fused ? dv.fac(Bt{}, 0) : T(0);
    for (int e0 = threadIdx.x; e0 < cells; e0 += 4 * blockDim.x) {
        T v[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int e = e0 + q * blockDim.x, y = e / nzp, z = e - y * nzp;
            v[q] = T(0);
            if (y < ny && z < nz) v[q] = fused ? dv.at(0, f, blockIdx.x, y, z) : src[(long)y * nz + z];
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int e = e0 + q * blockDim.x, y = e / nzp, z = e - y * nzp;
            if (e < cells) P[y * pz + z] = v[q];
        }
    }
    __syncthreads();
    acc_t acc[4];
    // z: Q[y][kz] = sum_m P[y][m] Cz[kz][m]; wave: column tile zt, row tiles
    // y0 .. y0 + ry - 1 (past the last: the last again, not stored)
    {
        const int zt = wave % tz, y0 = wave / tz * ry;
        const bool on = y0 < ty;
        const T* a = P + li * pz + lk;
        auto op = [&](int u, int k) { return a[16 * min(y0 + u, ty - 1) * pz + k]; };
        const T* O = Oz + (long)zt * tz * 256 + lane;
        if (on) {
            if (ry == 1) dw_contract<T, 1, false>(acc, O, 4 * tz, op);
            else if (ry == 2) dw_contract<T, 2, false>(acc, O, 4 * tz, op);
            else if (ry == 3) dw_contract<T, 3, false>(acc, O, 4 * tz, op);
            else dw_contract<T, 4, false>(acc, O, 4 * tz, op);
        }
        __syncthreads();   // the plane read by every wave
        if (on) {
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (u < ry && y0 + u < ty) {
#pragma unroll
                    for (int r = 0; r < 4; r++) P[(16 * (y0 + u) + Mma<T>::row(lk, r)) * pz + 16 * zt + li] = acc[u][r];
                }
        }
        __syncthreads();
    }
    // y: out[ky][kz] = sum_m Cy[ky][m] Q[m][kz]; wave: row tile yt, column
    // tiles z0 .. z0 + rz - 1
    const int yt = wave % ty, z0 = wave / ty * rz;
    if (z0 >= tz) return;
    const T* b = P + lk * pz + li;
    auto op = [&](int u, int k) { return b[k * pz + 16 * min(z0 + u, tz - 1)]; };
    const T* O = Oy + (long)yt * ty * 256 + lane;
    if (rz == 1) dw_contract<T, 1, true>(acc, O, 4 * ty, op);
    else if (rz == 2) dw_contract<T, 2, true>(acc, O, 4 * ty, op);
    else if (rz == 3) dw_contract<T, 3, true>(acc, O, 4 * ty, op);
    else dw_contract<T, 4, true>(acc, O, 4 * ty, op);
    const T norm = T(4 * po.ny * po.nz);
#pragma unroll
    for (int u = 0; u < 4; u++) {
        if (u >= rz || z0 + u >= tz) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int gm = 16 * yt + Mma<T>::row(lk, r), gn = 16 * (z0 + u) + li;
            if (gm >= ny || gn >= nz) continue;
            if (INV && po.phi) phi_store(po, (int)blockIdx.x, gm, gn, fdiv<T>(acc[u][r], norm));
            else io[blockIdx.x * plane + (long)gm * nz + gn] = acc[u][r];
        }
    }
}

// ------------------------------------------------- fast DCT of planes
//
// The (y, z) transforms of phisolver_dct for ny = nz = N, N = 128 or 256
// (fftw_3d.h REDFT10 forward, REDFT01 inverse, unnormalised) by Makhoul's
// reordering: a DCT-II of length N is the real part of a twiddled DFT of the
// even samples followed by the reversed odd ones, and that real-input DFT of
// length N is one complex DFT of length M = N/2 plus a split.  The complex
// DFT is four-step: M = 64 as 8 x 8 and M = 128 as 16 x 8 (radix-8 passes in
// registers, a twiddle, a transpose through LDS).  REDFT01 runs the same
// steps backwards.  Eight threads transform one line held in LDS.
// O(N log N) per line instead of the dense contractions' O(N^2), so a pass is
// a load and a store of HBM plus LDS work.  Twiddles for N (host double
// precision, rounded to T), as (cos, sin) pairs: tw[0 .. M-1] =
// e^{-2 pi i k/M}, tw[M .. M+N/2] = e^{-2 pi i k/N}, tw[N+1 .. 2N] =
// e^{-i pi k/(2N)}, 2N + 1 values.
constexpr int FD_N = 128, FD_P = 129;
constexpr int fd_tw_len(int n) { return 2 * n + 1; }

template <typename T>
struct Cx { T r, i; };
template <typename T>
__device__ __forceinline__ Cx<T> cmul(Cx<T> a, Cx<T> b) { return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r}; }
template <typename T>
__device__ __forceinline__ Cx<T> cconj(Cx<T> a) { return {a.r, -a.i}; }

// in-place 8-point DFT, natural order; INV uses e^{+2 pi i/8}
template <typename T, bool INV>
__device__ __forceinline__ void dft8(Cx<T> (&a)[8])
{
    const T h = T(0.70710678118654752440);
    Cx<T> s[4], d[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        s[j] = {a[j].r + a[j + 4].r, a[j].i + a[j + 4].i};
        d[j] = {a[j].r - a[j + 4].r, a[j].i - a[j + 4].i};
    }
    // d[j] *= w8^j
    const T sg = INV ? T(1) : T(-1);
    d[1] = {h * (d[1].r - sg * d[1].i), h * (d[1].i + sg * d[1].r)};
    d[2] = {-sg * d[2].i, sg * d[2].r};
    d[3] = {h * (-d[3].r - sg * d[3].i), h * (-d[3].i + sg * d[3].r)};
    Cx<T>* p[2] = {s, d};
#pragma unroll
    for (int q = 0; q < 2; q++) {
        Cx<T>* v = p[q];
        const Cx<T> s0 = {v[0].r + v[2].r, v[0].i + v[2].i}, d0 = {v[0].r - v[2].r, v[0].i - v[2].i};
        const Cx<T> s1 = {v[1].r + v[3].r, v[1].i + v[3].i};
        const Cx<T> t1 = {v[1].r - v[3].r, v[1].i - v[3].i};
        const Cx<T> d1 = {-sg * t1.i, sg * t1.r};   // t1 * w4
        a[q] = {s0.r + s1.r, s0.i + s1.i};
        a[q + 4] = {s0.r - s1.r, s0.i - s1.i};
        a[q + 2] = {d0.r + d1.r, d0.i + d1.i};
        a[q + 6] = {d0.r - d1.r, d0.i - d1.i};
    }
}

template <typename T>
__device__ __forceinline__ Cx<T> twl(const T* __restrict__ tw, int k) { return {tw[2 * k], tw[2 * k + 1]}; }

// in-place 16-point DFT as two 8-point DFTs (even, odd samples) and one
// radix-2 step; w16^k = tw[ws k] (the table's e^{-2 pi i k/M}, ws = M/16)
template <typename T, bool INV>
__device__ __forceinline__ void dft16(Cx<T> (&a)[16], const T* __restrict__ tw, int ws)
{
    Cx<T> e[8], o[8];
#pragma unroll
    for (int j = 0; j < 8; j++) { e[j] = a[2 * j]; o[j] = a[2 * j + 1]; }
    dft8<T, INV>(e);
    dft8<T, INV>(o);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        Cx<T> t = o[k];
        if (k > 0) {
            const Cx<T> w = twl(tw, ws * k);
            t = cmul(t, INV ? cconj(w) : w);
        }
        a[k] = {e[k].r + t.r, e[k].i + t.i};
        a[k + 8] = {e[k].r - t.r, e[k].i - t.i};
    }
}

// Position of real e of a line in LDS.  With SW (the 128 x 128 plane in
// LDS) bits 1..3 of e are XORed with bits 4..6: a permutation that keeps
// each complex value's two reals together and puts the values that the 8
// threads of a line touch at a stride of 16 reals (the transposed reads of
// fft_line) in different banks; without SW the line is in natural order.
template <bool SW>
__device__ __forceinline__ int lp(int e) { return SW ? (e ^ (((e >> 4) & 7) << 1)) : e; }

// complex value c of a line stored as reals (2c, 2c+1) at stride st
template <typename T, bool SW = false>
__device__ __forceinline__ Cx<T> lcx(const T* L, int st, int c)
{
    const int e = lp<SW>(2 * c);
    return {L[e * st], L[(e + 1) * st]};
}
template <typename T, bool SW = false>
__device__ __forceinline__ void scx(T* L, int st, int c, Cx<T> v)
{
    const int e = lp<SW>(2 * c);
    L[e * st] = v.r;
    L[(e + 1) * st] = v.i;
}

// M-point DFT (M = 64 or 128) of the line's complex values, in place
// through LDS, natural order in and out; thread t of the line's 8.  Four
// steps with M = P x 8: thread t takes the P values n = 8 n1 + t, DFTs them
// over n1, twiddles by e^{-2 pi i t k1/M} and stores at 8 k1 + t; then the
// 8-point DFTs over the contiguous 8 k1 .. 8 k1 + 7 (P/8 of them per thread)
// give X[k1 + P k2].  The line's 8 threads call it together (line_sync
// between the steps); the block's lines are independent of each other.
// The 8 threads of a line lie in one wave (consecutive thread indices), so
// their exchanges through LDS need the wave's accesses ordered, not the
// block's: a wave-scope fence on both sides of a wave barrier (the writes
// before it complete and are visible to the wave's reads after it).
__device__ __forceinline__ void line_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T, bool INV, int M, bool SW = false>
__device__ __forceinline__ void fft_line(T* L, int st, int t, const T* __restrict__ tw)
{
    static_assert(M == 64 || M == 128, "fft_line: M is 64 or 128");
    constexpr int P = M / 8;
    Cx<T> a[P];
#pragma unroll
    for (int n1 = 0; n1 < P; n1++) a[n1] = lcx<T, SW>(L, st, 8 * n1 + t);
    if constexpr (P == 8) dft8<T, INV>(a);
    else dft16<T, INV>(a, tw, M / 16);
#pragma unroll
    for (int k1 = 1; k1 < P; k1++) {
        const Cx<T> w = twl(tw, t * k1);
        a[k1] = cmul(a[k1], INV ? cconj(w) : w);
    }
    line_sync();
#pragma unroll
    for (int k1 = 0; k1 < P; k1++) scx<T, SW>(L, st, 8 * k1 + t, a[k1]);
    line_sync();
    Cx<T> b[P / 8][8];
#pragma unroll
    for (int g = 0; g < P / 8; g++) {
#pragma unroll
        for (int m2 = 0; m2 < 8; m2++) b[g][m2] = lcx<T, SW>(L, st, 8 * (t + 8 * g) + m2);
        dft8<T, INV>(b[g]);
    }
    line_sync();
#pragma unroll
    for (int g = 0; g < P / 8; g++)
#pragma unroll
        for (int k2 = 0; k2 < 8; k2++) scx<T, SW>(L, st, t + 8 * g + P * k2, b[g][k2]);
    line_sync();
}

// REDFT10 of one line of N reals at stride st, in place
template <typename T, int N, bool SW = false>
__device__ __forceinline__ void redft10_line(T* L, int st, int t, const T* __restrict__ tw)
{
    constexpr int M = N / 2, V = M / 8;
    // z[m] = v[2m] + i v[2m+1], v = even samples then reversed odd ones
    Cx<T> a[V];
#pragma unroll
    for (int m1 = 0; m1 < V; m1++) {
        const int m = 8 * m1 + t;
        a[m1] = m < N / 4 ? Cx<T>{L[lp<SW>(4 * m) * st], L[lp<SW>(4 * m + 2) * st]}
                          : Cx<T>{L[lp<SW>(2 * N - 1 - 4 * m) * st], L[lp<SW>(2 * N - 3 - 4 * m) * st]};
    }
    line_sync();
#pragma unroll
    for (int m1 = 0; m1 < V; m1++) scx<T, SW>(L, st, 8 * m1 + t, a[m1]);
    line_sync();
    fft_line<T, false, M, SW>(L, st, t, tw);
    // V[k] = (Z[k] + conj Z[M-k])/2 - i/2 WN^k (Z[k] - conj Z[M-k]);
    // X[k] = 2 Re(W4N^k V[k]), X[N-k] = -2 Im(W4N^k V[k])
    T xr[V + 1], xi[V + 1];
#pragma unroll
    for (int j = 0; j <= V; j++) {
        const int k = t + 8 * j;
        if (j < V || t == 0) {
            const Cx<T> zk = lcx<T, SW>(L, st, k & (M - 1)), zc = cconj(lcx<T, SW>(L, st, (M - k) & (M - 1)));
            const Cx<T> ve = {T(0.5) * (zk.r + zc.r), T(0.5) * (zk.i + zc.i)};
            const Cx<T> df = {zk.r - zc.r, zk.i - zc.i};
            const Cx<T> vo = {T(0.5) * df.i, T(-0.5) * df.r};   // -i/2 (Zk - Zc)
            const Cx<T> wv = cmul(twl(tw, M + k), vo);
            const Cx<T> v = {ve.r + wv.r, ve.i + wv.i};
            const Cx<T> q = cmul(twl(tw, N + 1 + k), v);
            xr[j] = T(2) * q.r;
            xi[j] = T(-2) * q.i;
        }
    }
    line_sync();
#pragma unroll
    for (int j = 0; j <= V; j++) {
        const int k = t + 8 * j;
        if (j < V || t == 0) {
            L[lp<SW>(k) * st] = xr[j];
            if (k >= 1 && k <= M - 1) L[lp<SW>(N - k) * st] = xi[j];
        }
    }
    line_sync();
}

// REDFT01 of one line of N reals at stride st, in place
template <typename T, int N, bool SW = false>
__device__ __forceinline__ void redft01_line(T* L, int st, int t, const T* __restrict__ tw)
{
    constexpr int M = N / 2, V = M / 8;
    // Vk = conj(W4N^k) (X[k] - i X[N-k]) (V0 = X[0]); c[k] = E + i O with
    // E = Vk + conj V(M-k), O = (Vk - conj V(M-k)) conj(WN^k)
    auto vk_of = [&](int k) -> Cx<T> {
        if (k == 0) return Cx<T>{L[0], T(0)};
        const Cx<T> x = {L[lp<SW>(k) * st], -L[lp<SW>(N - k) * st]};
        return cmul(cconj(twl(tw, N + 1 + k)), x);
    };
    Cx<T> c[V];
#pragma unroll
    for (int j = 0; j < V; j++) {
        const int k = t + 8 * j;
        const Cx<T> vk = vk_of(k), vh = cconj(vk_of(M - k));
        const Cx<T> e = {vk.r + vh.r, vk.i + vh.i};
        const Cx<T> o = cmul(Cx<T>{vk.r - vh.r, vk.i - vh.i}, cconj(twl(tw, M + k)));
        c[j] = {e.r - o.i, e.i + o.r};
    }
    line_sync();
#pragma unroll
    for (int j = 0; j < V; j++) scx<T, SW>(L, st, t + 8 * j, c[j]);
    line_sync();
    fft_line<T, true, M, SW>(L, st, t, tw);
    // y[2n] = v[n], y[2n+1] = v[N-1-n], v[2m] = Re z[m], v[2m+1] = Im z[m]
    Cx<T> z[V];
#pragma unroll
    for (int k2 = 0; k2 < V; k2++) z[k2] = lcx<T, SW>(L, st, t + 8 * k2);
    line_sync();
#pragma unroll
    for (int k2 = 0; k2 < V; k2++) {
        const int m = t + 8 * k2;
        if (m < N / 4) { L[lp<SW>(4 * m) * st] = z[k2].r; L[lp<SW>(4 * m + 2) * st] = z[k2].i; }
        else { L[lp<SW>(2 * N - 1 - 4 * m) * st] = z[k2].r; L[lp<SW>(2 * N - 3 - 4 * m) * st] = z[k2].i; }
    }
    line_sync();
}

// N = 128: the 2D transform of plane b in one block (the plane in LDS, row
// pitch 129): rows (z) then columns (y), 8 threads per line; the inverse
// writes phi (or out).  in may equal out: a block reads and writes only its
// own plane.
// Threads per block and layout of the plane transform, measured per
// precision: FP64 at 512 threads (two passes of 64 lines; at 1024 threads
// the 128-register limit per thread spills) with both transforms in lp
// order; FP32 at 1024 threads (one pass of 128 lines), the forward in
// natural order.
template <typename T> struct FdCfg {
    static constexpr int threads = sizeof(T) == 8 ? 512 : 1024;
    static constexpr bool sw_fwd = sizeof(T) == 8;
};

template <typename T, bool INV>
__global__ __launch_bounds__(FdCfg<T>::threads) void k_dct_plane(const T* in, T* out, const T* __restrict__ tw,
                                                                 PhiOut<T> po, DivIn<T> dv)
{
    constexpr int FD_THREADS = FdCfg<T>::threads;
    constexpr bool SW = INV || FdCfg<T>::sw_fwd;
    constexpr int LG = FD_THREADS / 8;   // lines transformed together
    extern __shared__ __align__(16) unsigned char pllc_smem[];
    T* pl = reinterpret_cast<T*>(pllc_smem);   // [128][FD_P]
    const int b = blockIdx.x, tid = threadIdx.x;
    const long base = (long)b * FD_N * FD_N;
    // point (y, z) of the plane sits at row lp(y), column lp(z) (lp the
    // identity without SW): every row and every column is a line in lp order
    if (!INV && dv.u) {
        const T f = dv.fac(Bt{}, 0);
#pragma unroll 4
        for (int e = tid; e < FD_N * FD_N; e += FD_THREADS)
            pl[lp<SW>(e >> 7) * FD_P + lp<SW>(e & 127)] = dv.at(0, f, b, e >> 7, e & 127);
    } else {
        for (int e = tid; e < FD_N * FD_N; e += FD_THREADS)
            pl[lp<SW>(e >> 7) * FD_P + lp<SW>(e & 127)] = in[base + e];
    }
    __syncthreads();
    const int t = tid & 7;
    for (int l0 = 0; l0 < FD_N; l0 += LG) {
        const int line = l0 + (tid >> 3);
        if (INV) redft01_line<T, FD_N, SW>(pl + line * FD_P, 1, t, tw);
        else redft10_line<T, FD_N, SW>(pl + line * FD_P, 1, t, tw);
    }
    __syncthreads();   // every row transformed before the columns are read
    for (int l0 = 0; l0 < FD_N; l0 += LG) {
        const int line = l0 + (tid >> 3);
        if (INV) redft01_line<T, FD_N, SW>(pl + line, FD_P, t, tw);
        else redft10_line<T, FD_N, SW>(pl + line, FD_P, t, tw);
    }
    __syncthreads();
    if (INV && po.phi) {
        const T norm = T(4 * po.ny * po.nz);
        for (int e = tid; e < FD_N * FD_N; e += FD_THREADS)
            phi_store(po, b, e >> 7, e & 127, fdiv<T>(pl[lp<SW>(e >> 7) * FD_P + lp<SW>(e & 127)], norm));
        return;
    }
    for (int e = tid; e < FD_N * FD_N; e += FD_THREADS) out[base + e] = pl[lp<SW>(e >> 7) * FD_P + lp<SW>(e & 127)];
}

// N = 128, FP32 data: the 2D transform of plane b as two dense contractions
// on the matrix cores in BF16x3 (each FP32 operand split as hi + lo, hi =
// bf16(x), lo = bf16(x - hi); a b ~ a_hi b_hi + a_hi b_lo + a_lo b_hi with
// FP32 accumulation, about 16 significant bits per product): first
// T = X Cz^T (z), then Y = Cy T (y), C the REDFT10 matrix (forward) or the
// REDFT01 matrix (inverse), stored as hi and lo BF16 arrays [out][in]
// (cb: fwd y, fwd z, inv y, inv z, each hi then lo).  The plane sits in LDS
// (row pitch DM_P); 8 waves, wave w owning rows 16 w .. 16 w + 15 of T and
// of Y.  v_mfma_f32_16x16x16_bf16: A 16 x 16 (lane l: row l % 16, columns
// 4 (l / 16) .. +3), B 16 x 16 (lane l: rows 4 (l / 16) .. +3, column
// l % 16), D (lane l: rows 4 (l / 16) .. +3, column l % 16).  Step one
// reads only the wave's own rows of X, so T overwrites them in place; the
// inverse writes phi normalised (and its face ghosts).  in may equal out.
constexpr int DM_N = 128, DM_P = 132;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short dm_bf4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float dm_f4;

__device__ __forceinline__ unsigned short dm_bf(float f)
{
    unsigned u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}
__device__ __forceinline__ void dm_split(const float (&x)[4], dm_bf4& hi, dm_bf4& lo)
{
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const unsigned short h = dm_bf(x[q]);
        hi[q] = (short)h;
        lo[q] = (short)dm_bf(x[q] - __uint_as_float((unsigned)h << 16));
    }
}

template <bool INV>
__global__ __launch_bounds__(512) void k_dct_bf16x3(const float* in, float* out,
                                                    const unsigned short* __restrict__ cb, PhiOut<float> po)
{
    extern __shared__ __align__(16) unsigned char pllc_smem[];
    float* pl = reinterpret_cast<float*>(pllc_smem);   // [128][DM_P]
    constexpr int N = DM_N, NN = DM_N * DM_N;
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const long base = (long)b * NN;
    for (int e = 4 * tid; e < NN; e += 4 * 512) {
        const float4 v = *(const float4*)(in + base + e);
        *(float4*)(pl + (e >> 7) * DM_P + (e & 127)) = v;
    }
    __syncthreads();
    const int m = lane & 15, kq = lane >> 4;
    const unsigned short* Cy = cb + (INV ? 4 : 0) * NN;   // hi, then lo at + NN
    const unsigned short* Cz = cb + (INV ? 6 : 2) * NN;
    {
        // T[y][k] = sum_z X[y][z] Cz[k][z], rows y of this wave
        dm_f4 acc[8];
#pragma unroll
        for (int t = 0; t < 8; t++) acc[t] = dm_f4{0.f, 0.f, 0.f, 0.f};
        const float* xr = pl + (16 * w + m) * DM_P + 4 * kq;
        for (int z0 = 0; z0 < N; z0 += 16) {
            const float4 xv = *(const float4*)(xr + z0);
            const float xa[4] = {xv.x, xv.y, xv.z, xv.w};
            dm_bf4 ah, al;
            dm_split(xa, ah, al);
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const long ci = (long)(16 * t + m) * N + z0 + 4 * kq;
                const dm_bf4 bh = *(const dm_bf4*)(Cz + ci), bl = *(const dm_bf4*)(Cz + NN + ci);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bh, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bl, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(al, bh, acc[t], 0, 0, 0);
            }
        }
#pragma unroll
        for (int t = 0; t < 8; t++)
#pragma unroll
            for (int q = 0; q < 4; q++) pl[(16 * w + 4 * kq + q) * DM_P + 16 * t + m] = acc[t][q];
    }
    __syncthreads();
    // Y[k'][k] = sum_y Cy[k'][y] T[y][k], rows k' of this wave
    dm_f4 acc[8];
#pragma unroll
    for (int t = 0; t < 8; t++) acc[t] = dm_f4{0.f, 0.f, 0.f, 0.f};
    for (int y0 = 0; y0 < N; y0 += 16) {
        const long ci = (long)(16 * w + m) * N + y0 + 4 * kq;
        const dm_bf4 ah = *(const dm_bf4*)(Cy + ci), al = *(const dm_bf4*)(Cy + NN + ci);
#pragma unroll
        for (int t = 0; t < 8; t++) {
            float tv[4];
#pragma unroll
            for (int q = 0; q < 4; q++) tv[q] = pl[(y0 + 4 * kq + q) * DM_P + 16 * t + m];
            dm_bf4 bh, bl;
            dm_split(tv, bh, bl);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bh, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bl, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(al, bh, acc[t], 0, 0, 0);
        }
    }
    if (INV && po.phi) {
        const float rn = 1.0f / float(4 * po.ny * po.nz);
#pragma unroll
        for (int t = 0; t < 8; t++)
#pragma unroll
            for (int q = 0; q < 4; q++) phi_store(po, b, 16 * w + 4 * kq + q, 16 * t + m, acc[t][q] * rn);
        return;
    }
#pragma unroll
    for (int t = 0; t < 8; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) out[base + (long)(16 * w + 4 * kq + q) * N + 16 * t + m] = acc[t][q];
}

// N = 256: a plane does not fit a block's LDS, so the 2D transform is two
// launches of FL lines per block (8 FL threads, 8 per line; LDS [FL][N + 1]):
// AX 2 transforms rows (z, contiguous): block B the packed rows FL B ..
// FL B + FL - 1; AX 1 transforms columns (y, stride N) of an FL-wide slab of
// z: block B plane B / (N/FL), z from FL (B % (N/FL)), staged as [z][y] so
// each column is a unit-stride LDS line.  The forward runs AX 2 then AX 1,
// the inverse AX 1 then AX 2, whose epilogue writes phi.  in may equal out:
// a block reads and writes only its own lines.  FL: 16 lines in FP64, 32 in
// FP32 (33 KB of LDS either way; measured fastest of 16 and 32 in each).
template <typename T>
constexpr int fl_lines() { return sizeof(T) == 8 ? 16 : 32; }
template <typename T, bool INV, int N, int AX, int FL>
__global__ __launch_bounds__(8 * FL) void k_dct_lines(const T* in, T* out, const T* __restrict__ tw, PhiOut<T> po,
                                                     DivIn<T> dv)
{
    extern __shared__ __align__(16) unsigned char pllc_smem[];
    T* ls = reinterpret_cast<T*>(pllc_smem);   // [FL][N + 1]
    constexpr int P = N + 1, E = FL * N, NT = 8 * FL;
    const int tid = threadIdx.x;
    const long blk = blockIdx.x;
    const long base = AX == 2 ? blk * E : (blk / (N / FL)) * N * N + (blk % (N / FL)) * FL;
    // element e of the block: its LDS slot and its offset from base
    auto slot = [&](int e) { return AX == 2 ? (e / N) * P + e % N : (e % FL) * P + e / FL; };
    auto goff = [&](int e) { return AX == 2 ? (long)e : (long)(e / FL) * N + e % FL; };
    constexpr int R = E / NT;   // values per thread
    {
        // every load of the thread in flight before the first LDS write
        T v[R];
        if (!INV && AX == 2 && dv.u) {
            const T f = dv.fac(Bt{}, 0);
            const int x = (int)(blk * FL / N), y0 = (int)(blk * FL % N);   // the block's rows lie in one plane
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int e = tid + NT * r;
                v[r] = dv.at(0, f, x, y0 + e / N, e % N);
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = in[base + goff(tid + NT * r)];
        }
#pragma unroll
        for (int r = 0; r < R; r++) ls[slot(tid + NT * r)] = v[r];
    }
    __syncthreads();
    const int line = tid >> 3, t = tid & 7;
    if (INV) redft01_line<T, N>(ls + line * P, 1, t, tw);
    else redft10_line<T, N>(ls + line * P, 1, t, tw);
    __syncthreads();   // the stores below read every line
    if (AX == 2 && INV && po.phi) {
        const T norm = T(4 * po.ny * po.nz);
#pragma unroll 2
        for (int q = 0; q < R; q++) {
            const int e = tid + NT * q;
            const long r = blk * FL + e / N;   // packed row b ny + gm
            phi_store(po, (int)(r / N), (int)(r % N), e % N, fdiv<T>(ls[slot(e)], norm));
        }
        return;
    }
#pragma unroll 4
    for (int q = 0; q < R; q++) out[base + goff(tid + NT * q)] = ls[slot(tid + NT * q)];
}

// ------------------------------------------------------------ utilities

// stream-ordered store of two device scalars, and with stale set the 16 stale
// values (k_stale) in the same launch
template <typename T>
__global__ void k_set_scalars(double* __restrict__ p, int i0, double v0, int i1, double v1, Dims d,
                              const T* __restrict__ q0, const T* __restrict__ q1, const T* __restrict__ q2,
                              const T* __restrict__ q3, T* __restrict__ stale)
{
    const int t = threadIdx.x;
    if (t == 0) { p[i0] = v0; p[i1] = v1; }
    if (stale && t < 16) stale[t] = stale_value<T>(d, q0, q1, q2, q3, t);
}

// rows of NZ values (grid.x blocks of (64, 4) threads over the rows): a field
// onto another, out of and into the contiguous FP64 rows of the host's arrays
template <typename T, typename F>
__device__ __forceinline__ void field_rows(const Dims& d, long rows, F f)
{
    for (long r = (long)blockIdx.x * blockDim.y + threadIdx.y; r < rows; r += (long)gridDim.x * blockDim.y)
        for (int k = threadIdx.x; k < d.NZ; k += 64) f(r * d.sy + k, r * d.NZ + k);
}
// b = a for the 12 (new, old) pairs (block row: the pair) in one launch: 56 us
// in 12 launches at 128x64x64 FP64, where a launch's floor is longer than a
// field's 4 MB
template <typename T>
struct CopyPairs { const T* a[12]; T* b[12]; };
template <typename T>
__global__ __launch_bounds__(256) void k_copy_pairs(Dims d, CopyPairs<T> cp, long rows)
{
    const T* __restrict__ a = cp.a[blockIdx.y];
    T* __restrict__ b = cp.b[blockIdx.y];
    field_rows<T>(d, rows, [&](long o, long) { b[o] = a[o]; });
}
template <typename T>
__global__ __launch_bounds__(256) void k_pack(Dims d, const T* __restrict__ a, double* __restrict__ b, long rows)
{
    field_rows<T>(d, rows, [&](long o, long l) { b[l] = double(a[o]); });
}
template <typename T>
__global__ __launch_bounds__(256) void k_unpack(Dims d, const double* __restrict__ a, T* __restrict__ b, long rows)
{
    field_rows<T>(d, rows, [&](long o, long l) { b[o] = T(a[l]); });
}

#ifdef PLLC_F64_TU
// ------------------------------------------------------------ diagnostics

// find_max (3539-3603) pass 1 over every point incl. ghosts: per block the
// last index of the largest |x| of each of u, v, w, c ("<=" keeps the later
// hit), and the first index where c.old, c.new or c.explicit_n is NaN.
__device__ __forceinline__ bool later_max(double b, long ib, double a, long ia)
{
    if (ib < 0) return false;
    if (ia < 0) return true;
    if (fabs(b) > fabs(a)) return true;
    if (fabs(b) < fabs(a)) return false;
    return ib > ia;
}

__global__ __launch_bounds__(256) void k_findmax_partial(long n, const double* __restrict__ u,
                                                         const double* __restrict__ v, const double* __restrict__ w,
                                                         const double* __restrict__ c, const double* __restrict__ co,
                                                         const double* __restrict__ cx, double* __restrict__ part)
{
    __shared__ double sv[4][256];
    __shared__ long si[4][256];
    __shared__ long snan[256];
    const int t = threadIdx.x;
    const double* q[4] = {u, v, w, c};
    double bv[4] = {0, 0, 0, 0};
    long bi[4] = {-1, -1, -1, -1};
    long nanat = -1;
    for (long l = (long)blockIdx.x * blockDim.x + t; l < n; l += (long)gridDim.x * blockDim.x) {
        for (int f = 0; f < 4; f++) {
            const double x = q[f][l];
            if (fabs(bv[f]) <= fabs(x) || bi[f] < 0) {
                if (!(x != x)) { bv[f] = x; bi[f] = l; }
            }
        }
        if (nanat < 0) {
            const double a1 = co[l], b1 = c[l], c1 = cx[l];
            if (a1 != a1 || b1 != b1 || c1 != c1) nanat = l;
        }
    }
    for (int f = 0; f < 4; f++) { sv[f][t] = bv[f]; si[f][t] = bi[f]; }
    snan[t] = nanat;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s) {
            for (int f = 0; f < 4; f++)
                if (later_max(sv[f][t + s], si[f][t + s], sv[f][t], si[f][t])) { sv[f][t] = sv[f][t + s]; si[f][t] = si[f][t + s]; }
            const long a = snan[t], b = snan[t + s];
            if (b >= 0 && (a < 0 || b < a)) snan[t] = b;
        }
        __syncthreads();
    }
    if (t == 0) {
        for (int f = 0; f < 4; f++) { part[blockIdx.x * 9 + 2 * f] = sv[f][0]; part[blockIdx.x * 9 + 2 * f + 1] = (double)si[f][0]; }
        part[blockIdx.x * 9 + 8] = (double)snan[0];
    }
}

// conc_average (3635-3728): y means per (i,k), z means per (i,j) and yz
// means per i of c over interior cells, each summed in the reference's
// order (one thread per output), divided as the reference divides.
__global__ void k_cavg(Dims d, const double* __restrict__ cn, float* __restrict__ ay, float* __restrict__ az,
                       float* __restrict__ ayz)
{
    const long nA = (long)d.nx * d.nz, nB = (long)d.nx * d.ny, nC = d.nx;
    long l = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (l < nA) {
        const int i = 3 + (int)(l / d.nz), k = 1 + (int)(l % d.nz);
        double s = 0;
        for (int j = 1; j <= d.ny; j++) s += cn[IX(d, i, j, k)];
        ay[l] = (float)(s / d.ny);
        return;
    }
    l -= nA;
    if (l < nB) {
        const int i = 3 + (int)(l / d.ny), j = 1 + (int)(l % d.ny);
        double s = 0;
        for (int k = 1; k <= d.nz; k++) s += cn[IX(d, i, j, k)];
        az[l] = (float)(s / d.nz);
        return;
    }
    l -= nB;
    if (l < nC) {
        const int i = 3 + (int)l;
        double s = 0;
        for (int j = 1; j <= d.ny; j++)
            for (int k = 1; k <= d.nz; k++) s += cn[IX(d, i, j, k)];
        ayz[l] = (float)(s / (d.ny * d.nz));
    }
}

// find_wmax (3606-3632): the largest w over interior cells (not |w|), >= 0
__global__ __launch_bounds__(256) void k_wmax(Dims d, const double* __restrict__ w, double* __restrict__ part)
{
    __shared__ double red[256];
    const int t = threadIdx.x;
    const long np = (long)d.nx * d.ny * d.nz;
    double m = 0.0;
    for (long l = (long)blockIdx.x * blockDim.x + t; l < np; l += (long)gridDim.x * blockDim.x) {
        const int i = 3 + (int)(l / ((long)d.ny * d.nz)), r = (int)(l % ((long)d.ny * d.nz));
        const double x = w[IX(d, i, 1 + r / d.nz, 1 + r % d.nz)];
        m = (x > m) ? x : m;
    }
    red[t] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s) red[t] = red[t + s] > red[t] ? red[t + s] : red[t];
        __syncthreads();
    }
    if (t == 0) part[blockIdx.x] = red[0];
}

void diag_findmax_partial(long n, const double* u, const double* v, const double* w, const double* c,
                          const double* co, const double* cx, double* part, int nb, hipStream_t st)
{
    k_findmax_partial<<<nb, 256, 0, st>>>(n, u, v, w, c, co, cx, part);
}

void diag_cavg(const Dims& d, const double* cn, float* ay, float* az, float* ayz, hipStream_t st)
{
    const long n = (long)d.nx * d.nz + (long)d.nx * d.ny + d.nx;
    k_cavg<<<(unsigned)((n + 127) / 128), 128, 0, st>>>(d, cn, ay, az, ayz);
}

void diag_wmax(const Dims& d, const double* w, double* part, int nb, hipStream_t st)
{
    k_wmax<<<nb, 256, 0, st>>>(d, w, part);
}
#endif  // PLLC_F64_TU

#ifdef PLLC_F64_TU
// batched single-line Thomas for the Tds entry points.  Element (line l,
// row i) of each array sits at l * ls + i * rs: the drop-in stages lines
// row-major (ls = 1, rs = nsys), so the 64 lanes of a wave read 64
// consecutive doubles of one row; line-major staging (ls = n, rs = 1) is
// accepted too.  mode 0 = tridiag_1rhs (b kept, solution in r, factors in
// cc), mode 1 = pll_tridiag (b, c overwritten as in pll_tridiag.c:21-47,
// cc unused).
__global__ void k_thomas_lines(int nsys, int n, long ls, long rs, const double* __restrict__ a,
                               double* __restrict__ b, double* __restrict__ c, double* __restrict__ r,
                               double* __restrict__ cc, int mode)
{
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= nsys) return;
    const long o = (long)l * ls;
    const double zero = 0.0;
    if (mode == 0) {
        double bb = b[o];
        cc[o] = c[o] / bb;
        r[o] = r[o] / bb;
        for (int i = 1; i < n; i++) {
            const long p = o + i * rs, q = p - rs;
            bb = b[p] - cc[q] * a[p];
            cc[p] = c[p] / bb;
            r[p] = (r[p] - r[q] * a[p]) / bb;
        }
        for (int i = n - 2; i >= 0; i--) {
            const long p = o + i * rs;
            r[p] = r[p] - r[p + rs] * cc[p];
        }
    } else {
        b[o] = b[o] - zero * a[o];
        c[o] = c[o] / b[o];
        r[o] = (r[o] - zero * a[o]) / b[o];
        for (int i = 1; i < n; i++) {
            const long p = o + i * rs, q = p - rs;
            b[p] = (b[p] - c[q] * a[p]);
            c[p] = c[p] / b[p];
            r[p] = (r[p] - r[q] * a[p]) / b[p];
        }
        const long e = o + (long)(n - 1) * rs;
        r[e] = r[e] - c[e] * zero;
        for (int i = n - 2; i >= 0; i--) {
            const long p = o + i * rs;
            r[p] = r[p] - c[p] * r[p + rs];
        }
    }
}

// calculate_weno for a batch of (kk, sign) positions on one D1 array
__global__ void k_weno_batch(const double* __restrict__ d1, const int* __restrict__ kk, const int* __restrict__ sg,
                             double* __restrict__ out, int n)
{
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= n) return;
    const int s = sg[l], b = kk[l];
    out[l] = weno5(d1[b], d1[b + s], d1[b + 2 * s], d1[b + 3 * s], d1[b + 4 * s]);
}

#endif  // PLLC_F64_TU

// ------------------------------------------------------ instantiations

#define PLLC_INST_RHS(T, FAST)                                                                                 \
    template __global__ void k_rhs<T, FAST>(Dims, Phys, RhsSets<T>, const T*, const T*, const T*, const T*,        \
                                            Visc4<T>, const T*, const T*, const T*, const double*, T, T, int, Bt);

#define PLLC_INST_DCT_PLANES(T, N)                                                                             \
    template __global__ void k_dct_planes<T, false, N>(int, int, int, int, T*, const T*, const T*, PhiOut<T>,  \
                                                       DivIn<T>, Bt);                                          \
    template __global__ void k_dct_planes<T, true, N>(int, int, int, int, T*, const T*, const T*, PhiOut<T>,   \
                                                      DivIn<T>, Bt);

#define PLLC_INST(T)                                                                                           \
    template __global__ void k_stale<T>(Dims, const T*, const T*, const T*, const T*, T*);                      \
    PLLC_INST_RHS(T, true)                                                                                     \
    PLLC_INST_RHS(T, false)                                                                                    \
    template __global__ void k_sweep<T, 0>(Dims, LineSets<T>, const double*, int, T, T);                      \
    template __global__ void k_sweep<T, 1>(Dims, LineSets<T>, const double*, int, T, T);                      \
    template __global__ void k_sweep<T, 2>(Dims, LineSets<T>, const double*, int, T, T);                      \
    template __global__ void k_sweep_z_lds<T>(Dims, LineSets<T>, const double*, T, T);                         \
    template __global__ void k_sweep_part<T, 0>(Dims, LineSets<T>, const double*, int, T, T, Bt);             \
    template __global__ void k_sweep_part<T, 1>(Dims, LineSets<T>, const double*, int, T, T, Bt);             \
    template __global__ void k_sweep_wave_z<T>(Dims, LineSets<T>, const double*, T, T, int, int, int, int, Bt); \
    template __global__ void k_visc<T>(Dims, Phys, const T*, T*, T*, T*, T*, Bt);                              \
    template __global__ void k_velo_ghost<T>(Dims, T*, T*, T*);                                                \
    template __global__ void k_phi_ghost<T>(Dims, T*);                                                         \
    template __global__ void k_div<T>(Dims, Phys, const T*, const T*, const T*, T*, T*, const double*, T, T);   \
    template __global__ void k_pack_div<T>(Dims, Phys, const T*, T*, const double*, T, T);                     \
    template __global__ void k_pois_x<T>(Dims, const T*, const T*, T*, T*, const double*);                     \
    template __global__ void k_velo_corr<T>(Dims, Phys, const T*, T*, T*, T*, const double*, T, T);            \
    template __global__ void k_flux_rows<T>(Dims, const T*, double*, Bt);                                      \
    template __global__ void k_flux_apply<T>(Dims, Phys, T*, double*, const double*, int, Bt);                 \
    template __global__ void k_pg<T>(Dims, Phys, Visc4<T>, const T*, T*, T*, T*, const double*, T, T, int);    \
    template __global__ void k_cfl_partial<T>(Dims, const T*, const T*, const T*, double*, Bt);                \
    template __global__ void k_bulk_partial<T>(Dims, const T*, double*);                                       \
    PLLC_INST_DCT_PLANES(T, 0)                                                                                 \
    PLLC_INST_DCT_PLANES(T, 16)                                                                                \
    PLLC_INST_DCT_PLANES(T, 32)                                                                                \
    PLLC_INST_DCT_PLANES(T, 48)                                                                                \
    PLLC_INST_DCT_PLANES(T, 64)                                                                                \
    template __global__ void k_dct_wide<T, false>(int, int, T*, const T*, const T*, PhiOut<T>, DivIn<T>);      \
    template __global__ void k_dct_wide<T, true>(int, int, T*, const T*, const T*, PhiOut<T>, DivIn<T>);       \
    template __global__ void k_gemm<T, true>(int, int, int, const T*, long, const T*, long, T*, long,          \
                                             PhiOut<T>);                                                        \
    template __global__ void k_gemm<T, false>(int, int, int, const T*, long, const T*, long, T*, long,         \
                                              PhiOut<T>);                                                       \
    template __global__ void k_dct_plane<T, false>(const T*, T*, const T*, PhiOut<T>, DivIn<T>);              \
    template __global__ void k_dct_plane<T, true>(const T*, T*, const T*, PhiOut<T>, DivIn<T>);               \
    template __global__ void k_dct_lines<T, false, 256, 1, fl_lines<T>()>(const T*, T*, const T*, PhiOut<T>, DivIn<T>); \
    template __global__ void k_dct_lines<T, false, 256, 2, fl_lines<T>()>(const T*, T*, const T*, PhiOut<T>, DivIn<T>); \
    template __global__ void k_dct_lines<T, true, 256, 1, fl_lines<T>()>(const T*, T*, const T*, PhiOut<T>, DivIn<T>); \
    template __global__ void k_dct_lines<T, true, 256, 2, fl_lines<T>()>(const T*, T*, const T*, PhiOut<T>, DivIn<T>); \
    template __global__ void k_copy_pairs<T>(Dims, CopyPairs<T>, long);                                        \
    template __global__ void k_pack<T>(Dims, const T*, double*, long);                                         \
    template __global__ void k_unpack<T>(Dims, const double*, T*, long);

// ------------------------------------------------- wave perturbation
//
// spline (pllcart3d.c:3280-3344) on lines of N points, in place: the
// natural spline's second derivatives from the (1,4,1) system of the
// interior points, solved with pll_tridiag's one-rank arithmetic
// (pll_tridiag.c:21-47), then evaluation at xx (or x - shift[k]) on the last
// interval holding it, with the reference's end rules (xx > x[N-1] takes
// y[N-1], xx < x[1] takes y[0]).  Line l starts at (l / nk) sj + (l % nk) sk,
// rows are rs apart; fp and cp are scratch with the same layout (cp also
// holds the new values until the line is rewritten).  One thread per line.
template <typename T>
__global__ void k_spline_lines(int N, long nlines, int nk, long sj, long sk, long rs, T delta,
                               const double* __restrict__ x, const double* __restrict__ xx,
                               const double* __restrict__ shift, T* __restrict__ y, T* __restrict__ cp,
                               T* __restrict__ fp)
{
    const long l = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= nlines) return;
    const long o = (l / nk) * sj + (l % nk) * sk;
    T* __restrict__ Y = y + o;
    T* __restrict__ C = cp + o;
    T* __restrict__ F = fp + o;
    const T zero = T(0.0), one = T(1.0), four = T(4.0);
    const int n = N - 2;
    auto rhs = [&](int i) {
        return T(6.0) / delta / delta * (Y[(long)(i + 1) * rs] - T(2.0) * Y[(long)i * rs] + Y[(long)(i - 1) * rs]);
    };
    // rows q = 0..n-1 (point i = q + 1) kept at line position i
    T b = four - zero * one;
    T c = one / b;
    T r = (rhs(1) - zero * one) / b;
    C[rs] = c;
    F[rs] = r;
    for (int q = 1; q < n; q++) {
        const long p = (long)(q + 1) * rs;
        b = (four - c * one);
        c = one / b;
        r = (rhs(q + 1) - r * one) / b;
        C[p] = c;
        F[p] = r;
    }
    r = r - c * zero;
    F[(long)n * rs] = r;
    for (int q = n - 2; q >= 0; q--) {
        const long p = (long)(q + 1) * rs;
        r = F[p] - C[p] * r;
        F[p] = r;
    }
    const T sh = shift ? T(shift[l % nk]) : zero;
    const T xl = T(x[N - 1]), x1 = T(x[1]);
    for (int ii = 0; ii < N; ii++) {
        const T xv = xx ? T(xx[ii]) : T(x[ii]) - sh;
        T v;
        if (xv > xl) v = Y[(long)(N - 1) * rs];
        else if (xv < x1) v = Y[0];
        else {
            // the largest i <= N-2 with x[i] <= xv (the reference's last hit)
            int lo = 1, hi = N - 2;
            while (lo < hi) {
                const int mid = (lo + hi + 1) / 2;
                if (T(x[mid]) <= xv) lo = mid;
                else hi = mid - 1;
            }
            const int i = lo;
            const T xi = T(x[i]), xi1 = T(x[i + 1]);
            const T fi = F[(long)i * rs];
            const T fi1 = (i + 1 == N - 1) ? zero : F[(long)(i + 1) * rs];
            v = fi * (xi1 - xv) * (xi1 - xv) * (xi1 - xv) / (T(6) * delta)
              + fi1 * (xv - xi) * (xv - xi) * (xv - xi) / (T(6) * delta)
              + (Y[(long)i * rs] / delta - delta / T(6) * fi) * (xi1 - xv)
              + (Y[(long)(i + 1) * rs] / delta - delta / T(6) * fi1) * (xv - xi);
        }
        C[(long)ii * rs] = v;
    }
    for (int ii = 0; ii < N; ii++) Y[(long)ii * rs] = C[(long)ii * rs];
}

// ------------------------------------------------ partitioned line solve
//
// The same systems as k_sweep, each line cut into P chunks of PM rows, one
// thread per chunk (the partition method for tridiagonal systems used by
// hybrid batched solvers).  A thread eliminates its chunk down to rows of the
// form A_t x_first + x_t + C_t x_last = D_t; its first and last rows couple
// only to the neighbouring chunks' boundary unknowns, a system solved by the
// line's threads together (PcrRow); every row then follows from its chunk's
// two boundary values.  Compared with one thread per line this gives P times
// the threads, keeps the eliminated rows in registers (no Thomas factors in
// HBM: S and mu are read once, the solution written once) and reads each row
// with one coalesced access per wavefront.  (I - fac A) is strictly
// diagonally dominant, so the result equals the Thomas solution to rounding.
//
// The kernels are bound by the latency of one chunk's instructions, so a
// chunk is straight code: all chunks have PM rows, a line's last chunk filled
// up with its last row again (they read the line's last row, whose upper
// coefficient is zero, so no row of the line reads them, and the coupling takes
// a zero first row after the last chunk), and boundary rows differ by
// numbers instead of branches.  (Chunks of varying length with their rows
// under conditions took 711 branches and 1700 integer instructions for the
// 650 FP64 operations of an x chunk, and one thread per line solving the
// coupling from LDS 2P dependent steps.)
constexpr int PM = 16;
constexpr int PART_THREADS = 512;    // threads per block of k_sweep_part at most
constexpr int POIS_THREADS = 1024;   // of k_pois_part

// keeps the scheduler from moving a chunk's rows into each other, which
// takes more registers than a wave has for them
__device__ __forceinline__ void row_done() { __builtin_amdgcn_sched_barrier(0); }

// the same offset with its origin hidden from the compiler, which otherwise
// keeps the 16 addresses of a chunk's loads in registers (32 of them) for
// the stores after the solve
__device__ __forceinline__ long renew(long o)
{
    asm volatile("" : "+v"(o));
    return o;
}

// a line's rows of one chunk: row t is -k_t x_{t-1} + (1 + k_t + k_{t+1}) x_t
// - k_{t+1} x_{t+1} = sv[t], k_t = kf mv[t], kf = fac del / h, mv the
// viscosity (1 for c).  The line's last row is row tl (PM or more: in a later
// chunk), its upper coefficient k_{tl+1} counted e1 times in the diagonal and
// dropped; first: row 0 is the line's first, its k_0 counted e0 times and
// dropped.  Rows past tl hold anything finite: they read row tl, no row reads
// them.
template <typename T>
struct PRows {
    T sv[PM], mv[PM + 1], kf, e0, e1;
    int tl;
    bool first;
};

// the factor of a boundary row's outer coefficient in its diagonal: Neumann
// b += off, Dirichlet b -= off (apply_bc) with off = -k
template <typename T>
__device__ __forceinline__ T bc_factor(int kind)
{
    return kind == BC_NEU ? T(0.0) : kind == BC_DIR ? T(2.0) : T(1.0);
}

template <typename T>
struct PChunk {
    T A[PM], C[PM], D[PM];

    // row t: a x_{t-1} + b x_t + c x_{t+1} = d (rows in order)
    __device__ __forceinline__ void fwd(int t, T a, T b, T c, T d)
    {
        if (t < 2) {
            const T rb = prcp<T>(b);
            D[t] = d * rb; A[t] = a * rb; C[t] = c * rb;
        } else {
            const T rb = prcp<T>(b - a * C[t - 1]);
            D[t] = rb * (d - a * D[t - 1]);
            A[t] = -rb * a * A[t - 1];
            C[t] = rb * c;
        }
    }

    // the backward pass and the first row's fold; leaves the chunk's outer
    // rows in A/C/D[0] and A/C/D[PM - 1]
    __device__ __forceinline__ void fold()
    {
#pragma unroll
        for (int t = PM - 3; t >= 1; t--) {
            D[t] = D[t] - C[t] * D[t + 1];
            A[t] = A[t] - C[t] * A[t + 1];
            C[t] = -C[t] * C[t + 1];
            row_done();
        }
        const T rb = prcp<T>(T(1.0) - C[0] * A[1]);
        D[0] = rb * (D[0] - C[0] * D[1]);
        A[0] = rb * A[0];
        C[0] = -rb * C[0] * C[1];
    }

    // the chunk's solution from its boundary values, in D
    __device__ __forceinline__ void solve(T xf, T xl)
    {
        D[0] = xf;
#pragma unroll
        for (int t = 1; t < PM - 1; t++) D[t] = D[t] - A[t] * xf - C[t] * xl;
        D[PM - 1] = xl;
    }
};

template <typename T>
__device__ __forceinline__ void chunk_rows(PChunk<T>& ch, const PRows<T>& r)
{
    T k0 = r.kf * r.mv[0];
#pragma unroll
    for (int t = 0; t < PM; t++) {
        const T k1 = r.kf * r.mv[t + 1];
        const bool end = t == r.tl;
        T a = -k0, kb = k0;
        if (t == 0) {
            kb = (r.first ? r.e0 : T(1.0)) * k0;
            a = r.first ? T(0.0) : a;
        }
        const T b = T(1.0) + kb + (end ? r.e1 * k1 : k1);
        ch.fwd(t, a, b, end ? T(0.0) : -k1, r.sv[t]);
        k0 = k1;
        row_done();
    }
    ch.fold();
}

// A chunk's share of its line's coupling.  The first row is A0 x_last(s-1) +
// x_first + C0 x_last = D0, the last Al x_first + x_last + Cl x_first(s+1) =
// Dl; with the first rows eliminated the P last unknowns form a tridiagonal
// system of unit diagonal, a x_last(s-1) + x_last + c x_last(s+1) = d, solved
// by parallel cyclic reduction: log2(P) rounds in which row s takes rows
// s -/+ w, w = 1, 2, 4, ..., zero outside the line.
template <typename T>
struct PcrRow {
    T a, c, d;
    // An, Cn, Dn: the next chunk's first row (zero after the last chunk)
    __device__ __forceinline__ void start(const PChunk<T>& ch, T An, T Cn, T Dn)
    {
        const T Al = ch.A[PM - 1], Cl = ch.C[PM - 1];
        const T r = prcp<T>(T(1.0) - Al * ch.C[0] - Cl * An);
        a = -(Al * ch.A[0]) * r;
        c = -(Cl * Cn) * r;
        d = (ch.D[PM - 1] - Al * ch.D[0] - Cl * Dn) * r;
    }
    __device__ __forceinline__ void round(T am, T cm, T dm, T ap, T cp, T dp)
    {
        const T r = prcp<T>(T(1.0) - a * cm - c * ap);
        d = (d - a * dm - c * dp) * r;
        a = -(a * am) * r;
        c = -(c * cp) * r;
    }
};

// the coupling through LDS, for lines whose chunks are threads s = 0 .. P-1
// of a block at the same q: two sets of [3][P][LPB] values read and written
// in turn, so a round needs one barrier.  Every thread of the block calls it
// (dead threads, without a line, only keep the barriers).
template <typename T>
__device__ __forceinline__ void chunk_couple(T* __restrict__ buf, int P, int LPB, int q, int s, bool live,
                                             PChunk<T>& ch)
{
    const int PL = P * LPB, o = s * LPB + q;
    T* cur = buf;
    T* nxt = buf + 3 * PL;
    if (live) {
        cur[o] = ch.A[0];
        cur[PL + o] = ch.C[0];
        cur[2 * PL + o] = ch.D[0];
    }
    __syncthreads();
    PcrRow<T> w;
    if (live) {
        const bool in = s + 1 < P;
        const int e = in ? o + LPB : o;
        const T An = cur[e], Cn = cur[PL + e], Dn = cur[2 * PL + e];
        w.start(ch, in ? An : T(0.0), in ? Cn : T(0.0), in ? Dn : T(0.0));
        nxt[o] = w.a;
        nxt[PL + o] = w.c;
        nxt[2 * PL + o] = w.d;
    }
    __syncthreads();
    for (int k = 1; k < P; k <<= 1) {
        T* t = cur;
        cur = nxt;
        nxt = t;
        if (live) {
            const bool lo = s >= k, hi = s + k < P;
            const int el = lo ? o - k * LPB : o, eh = hi ? o + k * LPB : o;
            const T am = cur[el], cm = cur[PL + el], dm = cur[2 * PL + el];
            const T ap = cur[eh], cp = cur[PL + eh], dp = cur[2 * PL + eh];
            w.round(lo ? am : T(0.0), lo ? cm : T(0.0), lo ? dm : T(0.0), hi ? ap : T(0.0), hi ? cp : T(0.0),
                    hi ? dp : T(0.0));
            nxt[o] = w.a;
            nxt[PL + o] = w.c;
            nxt[2 * PL + o] = w.d;
        }
        __syncthreads();
    }
    if (live) {
        const T xp = s > 0 ? nxt[2 * PL + o - LPB] : T(0.0);
        ch.solve(ch.D[0] - ch.C[0] * w.d - ch.A[0] * xp, w.d);
    }
}

// lanes per row of the x- and y-sweeps
__host__ __device__ constexpr int line_row(int nz) { return (nz + 15) / 16 * 16; }

// x- and y-lines (rows strided by sx / sy): block (LPB lines along k,
// P chunks); a wavefront reads one row of consecutive k, coalesced.  At most
// 128 registers (q_old is read after the coupling), so that in FP64 two
// blocks of 512 threads share a CU.  Measured, u, v and w in one launch, with
// branches and a serial coupling before: 256x128x128 x 117 -> 83 us FP64
// (5.1 TB/s of S, mu, q_old, q_new), 59 -> 40 mixed, y 63 -> 57 and 35 -> 27;
// 512x256x256 x 1110 -> 750 and 552 -> 422, y 475 -> 473 (5.3 TB/s) and 257 ->
// 232; 64x32x32 (latency) x 11.6 -> 9.1, y 8.1 -> 5.3
template <typename T, int DIR>
__global__ __launch_bounds__(PART_THREADS, 4) void k_sweep_part(Dims d, LineSets<T> sets, const double* __restrict__ scal,
                                                       int slot, T g, T r, Bt bt)
{
    extern __shared__ unsigned char pllc_smem[];
    T* red = reinterpret_cast<T*>(pllc_smem);
    const int LPB = blockDim.x, q = threadIdx.x, s = threadIdx.y;
    // member: blockIdx.z
    const LineSet<T> L = bt_lines<T, DIR>(bt, sets.s[blockIdx.y], blockIdx.z);
    scal += blockIdx.z * S_SIZE;
    const Rng R = L.R;
    // Lanes cover k = 1 .. nz of a row, rounded up to 16 lanes (an aligned
    // piece of a pitched one).  x-lines: the y ghosts of the new values (jg) are rows of
    // lanes of their own that solve the line next to the wall again and store
    // at their own place; the z ghosts (kg) are stored by the lanes at the
    // row's ends
    const int jg = DIR == 0 && L.jg;
    const int n0 = line_row(d.nz);
    const int n1 = DIR == 0 ? R.je - R.js + 1 + 2 * jg : R.ie - R.is + 1;
    // blocks of one line set: grid x is a multiple of 8 (XCD order within the set)
    const int bx = (gridDim.x & 7) == 0 ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    const int l = bx * LPB + q;
    const int n = DIR == 0 ? R.ie - R.is + 1 : R.je - R.js + 1;
    const int x0 = s * PM;
    const int a1 = l / n0, kl = l - a1 * n0 + 1;
    // a set with shorter lines than the launch's longest may need fewer chunks
    const bool live = x0 < n && a1 < n1 && kl >= R.ks && kl <= R.ke;
    const int k = live ? kl : R.ks;
    const int jl = R.js - jg + a1;   // x-lines: the lane's place
    int i, j;
    long st;
    if (DIR == 0) { j = live ? min(max(jl, R.js), R.je) : R.js; i = R.is; st = d.sx; }
    else { i = live ? R.is + a1 : R.is; j = R.js; st = d.sy; }
    const bool own = DIR != 0 || j == jl;   // not a ghost lane
    const bool last = x0 + PM >= n;
    const int nv = min(PM, n - x0);
    const long o0 = IX(d, i, j, k) + (long)(live ? x0 : 0) * st;
    const T* __restrict__ S = L.S + o0;
    const bool cst = L.mu == nullptr;
    const T dt = T(scal[S_DT]);
    const T fac = T(0.5) * dt * (g + r);

    PChunk<T> ch;
    if (live) {
        PRows<T> w;
        w.tl = nv - 1;
        if (!last) w.tl = PM;
        // past the line's end: its last row (and the mu above it) again
        const T* __restrict__ mu = cst ? nullptr : L.mu + o0 + L.mu_off;
        if (nv == PM) {
#pragma unroll
            for (int t = 0; t < PM; t++) w.sv[t] = S[(long)t * st];
            if (!cst) {
#pragma unroll
                for (int t = 0; t <= PM; t++) w.mv[t] = mu[(long)t * st];
            }
        } else {
            const int si = (int)st;
            const unsigned lim = (nv - 1) * si;
#pragma unroll
            for (int t = 0; t < PM; t++) w.sv[t] = S[min((unsigned)(t * si), lim)];
            if (!cst) {
#pragma unroll
                for (int t = 0; t <= PM; t++) w.mv[t] = mu[min((unsigned)(t * si), lim + si)];
            }
        }
        if (cst) {
#pragma unroll
            for (int t = 0; t <= PM; t++) w.mv[t] = T(1.0);
        }
        w.kf = cst ? fac * L.ca : fac * L.del * T(L.rh);
        w.first = s == 0;
        w.e0 = bc_factor<T>(L.bc0);
        w.e1 = DIR == 0 ? T(1.0) : bc_factor<T>(L.bc1);
        if (DIR == 0 && last) {
            // explicit outflow face iend+1 (677-683 and matching lines)
            const long ob = o0 + (long)nv * st;
            const T vbulk = T(scal[S_RK + 4 * slot]);
            const T q1 = L.qold[ob], q0 = L.qold[ob - st], n1o = L.Nm1[ob];
            const T mtop = cst ? T(1.0) : mu[(long)nv * st];
            const T nb = divh<T>(-vbulk * (q1 - q0), T(d.dx), d.rdx);
            const T bcor = dt * (g * nb + r * n1o);
            if (own) {
                L.N[ob] = nb;
                L.qnew[ob] = q1 + bcor;
            }
            const T radd = w.kf * mtop * bcor;
#pragma unroll
            for (int t = 0; t < PM; t++) w.sv[t] += t == w.tl ? radd : T(0.0);
        }
        chunk_rows<T>(ch, w);
    }
    chunk_couple<T>(red, (n + PM - 1) / PM, LPB, q, s, live, ch);
    if (!live) return;
    const long on = renew(o0);
    if (DIR == 1) {
        T* so = L.S + on;
        if (nv == PM) {
#pragma unroll
            for (int t = 0; t < PM; t++) so[(long)t * st] = ch.D[t];
        } else {
#pragma unroll
            for (int t = 0; t < PM; t++)
                if (t < nv) so[(long)t * st] = ch.D[t];
        }
        return;
    }
    // c's ghosts are copies (700-712; the y-ghost rows' z ghosts too), the
    // velocities' z ghosts copies, their y ghosts negated, their corners
    // never written (velo_ghost_point)
    const bool vel = L.F != FC;
    const T sg = vel && !own ? T(-1.0) : T(1.0);
    const T* qo = L.qold + on;
    T* qn = L.qnew + on + (long)(jl - j) * d.sy;
    if (nv == PM) {
        T v[PM];
#pragma unroll
        for (int t = 0; t < PM; t++) v[t] = qo[(long)t * st];
#pragma unroll
        for (int t = 0; t < PM; t++) {
            ch.D[t] = sg * (v[t] + ch.D[t]);
            qn[(long)t * st] = ch.D[t];
        }
    } else {
#pragma unroll
        for (int t = 0; t < PM; t++)
            if (t < nv) {
                ch.D[t] = sg * (qo[(long)t * st] + ch.D[t]);
                qn[(long)t * st] = ch.D[t];
            }
    }
    if (L.kg && (own || !vel) && (k == R.ks || k == R.ke)) {
        for (int e = -1; e <= 1; e += 2) {
            if (k != (e < 0 ? R.ks : R.ke)) continue;
#pragma unroll
            for (int t = 0; t < PM; t++)
                if (t < nv) qn[(long)t * st + e] = ch.D[t];
        }
    }
    // the inlet ghosts of v and w
    if (s == 0 && own && L.inlet) qn[-d.sx] = -ch.D[0];
}

// value of x moved by W lanes within its row of 16 lanes (UP: from the lane
// W below), by a DPP move; zero where that lies outside the row
template <int W, bool UP>
__device__ __forceinline__ int dpp_shift(int x)
{
    return __builtin_amdgcn_update_dpp(0, x, (UP ? 0x110 : 0x100) + W, 0xf, 0xf, true);
}
template <int W, bool UP>
__device__ __forceinline__ float lane_shift(float x)
{
    return __int_as_float(dpp_shift<W, UP>(__float_as_int(x)));
}
template <int W, bool UP>
__device__ __forceinline__ double lane_shift(double x)
{
    return __hiloint2double(dpp_shift<W, UP>(__double2hiint(x)), dpp_shift<W, UP>(__double2loint(x)));
}

// one round of the coupling between lanes W apart, lane g of a line's P.
// ROW: the line's lanes lie in one row of 16 (DPP moves); else ds_bpermute.
template <typename T, int W, bool ROW>
__device__ __forceinline__ void lane_round(PcrRow<T>& w, int g, int P)
{
    const bool lo = g >= W, hi = g + W < P;
    T am, cm, dm, ap, cp, dp;
    if constexpr (ROW) {
        am = lane_shift<W, true>(w.a); cm = lane_shift<W, true>(w.c); dm = lane_shift<W, true>(w.d);
        ap = lane_shift<W, false>(w.a); cp = lane_shift<W, false>(w.c); dp = lane_shift<W, false>(w.d);
    } else {
        am = __shfl_up(w.a, W); cm = __shfl_up(w.c, W); dm = __shfl_up(w.d, W);
        ap = __shfl_down(w.a, W); cp = __shfl_down(w.c, W); dp = __shfl_down(w.d, W);
    }
    w.round(lo ? am : T(0.0), lo ? cm : T(0.0), lo ? dm : T(0.0), hi ? ap : T(0.0), hi ? cp : T(0.0),
            hi ? dp : T(0.0));
}

// z-lines (rows contiguous along k).  A wave owns 64 chunks: 64 / G lines of
// one i-plane and one line set (consecutive j), G lanes per line, G the power
// of two of at least the P chunks of a line.  The rows pass through the
// wave's own LDS tile (coalesced in HBM, by chunk in registers; slot 17 g +
// t holds row 16 g + t, so the lanes' chunk reads fall in distinct banks and
// slot 17 g + 16 is free), S first, then mu in the same slots, then the
// solution; the coupling runs between lanes.  Waves are independent of each
// other: no block barriers, so the loads, eliminations and stores of a CU's
// waves overlap.  Bound by HBM in both precisions: u, v and w at 256x128x128
// 56 us FP64 (5.7 TB/s of S, mu, S) and 28 us mixed, where a tile per block
// with the rows' loads, eliminations and stores between block barriers took
// 90 and 51; at 512x256x256 480 and 229 us against 790 and 325; at 64x32x32
// 7.1 against 12.  (FP64 at 4 waves per SIMD spills: 64 us.)  nbx: tiles per
// plane; ntiles: tiles of all planes and sets
// of a member.
constexpr int ZW = 17;                    // LDS slots per chunk
constexpr int Z_TILE = 64 * ZW;           // per wave
constexpr int Z_WAVES = 4;                // waves per block at most

template <typename T>
__global__ __launch_bounds__(64 * Z_WAVES, sizeof(T) == 8 ? 3 : 4) void k_sweep_wave_z(Dims d, LineSets<T> sets,
                                                                  const double* __restrict__ scal, T g, T r, int G,
                                                                  int nbx, int ni, int ntiles, Bt bt)
{
    extern __shared__ __align__(16) unsigned char pllc_smem[];
    const int lane = threadIdx.x & 63;
    T* ls = reinterpret_cast<T*>(pllc_smem) + (threadIdx.x >> 6) * Z_TILE;
    const int mb = blockIdx.y;   // member
    // XCD x takes the x-th eighth of the blocks: neighbouring tiles share
    // cache lines at their edges
    const int bx = (gridDim.x & 7) == 0 ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    const int tile = __builtin_amdgcn_readfirstlane(bx * (blockDim.x >> 6) + (threadIdx.x >> 6));
    if (tile >= ntiles) return;
    const int per_set = nbx * ni, set = tile / per_set, rem = tile - set * per_set;
    const int ii = rem / nbx, jb = rem - ii * nbx;
    const LineSet<T> L = bt_lines<T, 2>(bt, sets.s[set], mb);
    scal += mb * S_SIZE;
    const Rng R = L.R;
    const int n = R.ke - R.ks + 1, LW = 64 / G;
    const int i = R.is + ii, j0 = R.js + jb * LW;
    const int nl = min(LW, R.je - j0 + 1);
    if (i > R.ie || nl <= 0) return;
    const int P = (n + PM - 1) / PM;
    const long base = IX(d, i, j0, R.ks);
    const bool cst = L.mu == nullptr;
    // element m of the lane: e = lane + 64 m of the tile's LW x 16 G slots,
    // row e % (16 G) of line e / (16 G): a lane's part and a part of m alone
    const int W = PM * G, lw = __builtin_ctz(W);
    const int xl = lane & (W - 1), ll = lane >> lw;
    const int ml = ll * G * ZW + xl + (xl >> 4);
    auto xs = [&](int m) { return (64 * m) & (W - 1); };
    auto rs = [&](int m) { return (64 * m) >> lw; };
    auto slot = [&](int m) { return ml + rs(m) * G * ZW + xs(m) + (xs(m) >> 4); };
    const bool exact = n == W && nl == LW;   // every slot is an element
    // past the line's end (xe: its last element to be read) or the last
    // line: its last element again
    auto load = [&](const T* __restrict__ p, int xe, T (&v)[PM]) {
        if (exact) {
            const T* __restrict__ pl = p + (long)ll * d.sy + xl;
#pragma unroll
            for (int m = 0; m < PM; m++) v[m] = pl[(long)rs(m) * d.sy + xs(m)];
        } else {
#pragma unroll
            for (int m = 0; m < PM; m++)
                v[m] = p[min(ll + rs(m), nl - 1) * (unsigned)d.sy + min(xl + xs(m), xe)];
        }
    };
    T vs[PM], vm[PM], mt = T(1.0);
    load(L.S + base, n - 1, vs);
    const int q = lane / G, c = lane - q * G;   // the lane's line and chunk
    if (!cst) {
        const T* __restrict__ mu = L.mu + L.mu_off + base;
        load(mu, n, vm);
        // the value above the last row has no slot in a line of 16 G rows
        mt = mu[(long)min(q, nl - 1) * d.sy + n];
    }
    T* mine = ls + lane * ZW;
#pragma unroll
    for (int m = 0; m < PM; m++) ls[slot(m)] = vs[m];
    line_sync();
    PRows<T> w;
#pragma unroll
    for (int t = 0; t < PM; t++) w.sv[t] = mine[t];
    const T fac = T(0.5) * T(scal[S_DT]) * (g + r);
    w.tl = n - c * PM - 1;
    w.first = c == 0;
    w.e0 = bc_factor<T>(L.bc0);
    w.e1 = bc_factor<T>(L.bc1);
    if (cst) {
#pragma unroll
        for (int t = 0; t <= PM; t++) w.mv[t] = T(1.0);
    } else {
        line_sync();
#pragma unroll
        for (int m = 0; m < PM; m++) ls[slot(m)] = vm[m];
        line_sync();
#pragma unroll
        for (int t = 0; t < PM; t++) w.mv[t] = mine[t];
        w.mv[PM] = mine[c == G - 1 ? PM - 1 : ZW];
        if (c == G - 1) w.mv[PM] = mt;
    }
    w.kf = cst ? fac * L.ca : fac * L.del * T(L.rh);
    PChunk<T> ch;
    chunk_rows<T>(ch, w);
    PcrRow<T> p;
    const bool nx = c + 1 < P;
    const T An = __shfl_down(ch.A[0], 1), Cn = __shfl_down(ch.C[0], 1), Dn = __shfl_down(ch.D[0], 1);
    p.start(ch, nx ? An : T(0.0), nx ? Cn : T(0.0), nx ? Dn : T(0.0));
    if (G <= 16) {
        if (P > 1) lane_round<T, 1, true>(p, c, P);
        if (P > 2) lane_round<T, 2, true>(p, c, P);
        if (P > 4) lane_round<T, 4, true>(p, c, P);
        if (P > 8) lane_round<T, 8, true>(p, c, P);
    } else {
        lane_round<T, 1, false>(p, c, P);
        lane_round<T, 2, false>(p, c, P);
        lane_round<T, 4, false>(p, c, P);
        lane_round<T, 8, false>(p, c, P);
        lane_round<T, 16, false>(p, c, P);
        if (P > 32) lane_round<T, 32, false>(p, c, P);
    }
    const T xp = __shfl_up(p.d, 1);
    ch.solve(ch.D[0] - ch.C[0] * p.d - ch.A[0] * (c > 0 ? xp : T(0.0)), p.d);
    line_sync();
#pragma unroll
    for (int t = 0; t < PM; t++) mine[t] = ch.D[t];
    line_sync();
    T* So = L.S + renew(base) + (long)ll * d.sy + xl;
    if (exact) {
#pragma unroll
        for (int m = 0; m < PM; m++) vs[m] = ls[slot(m)];
#pragma unroll
        for (int m = 0; m < PM; m++) So[(long)rs(m) * d.sy + xs(m)] = vs[m];
    } else {
#pragma unroll
        for (int m = 0; m < PM; m++)
            if (xl + xs(m) < n && ll + rs(m) < nl) So[(long)rs(m) * d.sy + xs(m)] = ls[slot(m)];
    }
}

// Poisson x-lines (phisolver_dct's pll_tridiag, 2055-2100) by the same
// partition method: line l = (y mode, z mode) of the packed block, rows x
// nm = ny nz apart, a = c = 1/dx^2, b = -2/dx^2 + lam_y + lam_z, Neumann
// rows at the inlet and (all modes but the mean) at the outlet.
//
// The mean mode (0,0), the gauge line of the otherwise singular problem, has
// lam = 0, Neumann at the inlet and the ghost phi = 0 at the outlet: its
// differences phi_{i+1} - phi_i are dx^2 times the sum of the sources up to
// i, and phi_i minus the sum of those from i on.  A block of its own forms
// the two sums in FP64 whatever the field type, each thread over consecutive
// rows with a scan over the threads between, so that the FP32 kernel holds
// no FP64 chunk (which cost it 166 registers).  Measured (FP64, mixed):
// 256x128x128 28 -> 15 us and 25 -> 11.5; 512x256x256, whose 32 chunks per
// line left 8 lines (64 or 32 bytes of a row) per block of 256 threads, 173
// -> 86 and 179 -> 57; 64x32x32 14 -> 4.8.
template <typename T>
__device__ __forceinline__ void pois_mean(const Dims& d, T* __restrict__ p, long nm, double* __restrict__ sh, int t,
                                          int NT)
{
    const int n = d.nx;
    const int x0 = (int)((long)t * n / NT), x1 = (int)((long)(t + 1) * n / NT);
    const double h2 = d.dx * d.dx;
    // inclusive scan of v over the block's threads (up: t ascending)
    auto scan = [&](double v, bool up) {
        double* cur = sh;
        double* nxt = sh + NT;
        cur[t] = v;
        __syncthreads();
        for (int w = 1; w < NT; w <<= 1) {
            if (up) { if (t >= w) v += cur[t - w]; }
            else { if (t + w < NT) v += cur[t + w]; }
            nxt[t] = v;
            __syncthreads();
            double* q = cur;
            cur = nxt;
            nxt = q;
        }
        __syncthreads();
        return v;
    };
    double f = 0.0;
    for (int x = x0; x < x1; x++) f += double(p[(long)x * nm]);
    const double before = scan(f, true) - f;   // the sources of the rows before x0
    double acc = before, g = 0.0;
    for (int x = x0; x < x1; x++) {
        acc += double(p[(long)x * nm]);
        g += h2 * acc;
    }
    double phi = -(scan(g, false) - g);   // phi of row x1
    // the segment again from its last row: acc is the sum up to row x
    for (int x = x1 - 1; x >= x0; x--) {
        const double s = double(p[(long)x * nm]);
        phi -= h2 * acc;
        acc -= s;
        p[(long)x * nm] = T(phi);
    }
}

template <typename T>
__global__ __launch_bounds__(POIS_THREADS, 4) void k_pois_part(Dims d, const T* __restrict__ lam_y, const T* __restrict__ lam_z,
                                                      T* __restrict__ P, Bt bt)
{
    extern __shared__ __align__(8) unsigned char pllc_smem[];
    // member: blockIdx.y
    P += blockIdx.y * bt.pk;
    const int LPB = blockDim.x, PC = blockDim.y;
    const int q = threadIdx.x, s = threadIdx.y;
    const long nm = (long)d.ny * d.nz;
    if (blockIdx.x == gridDim.x - 1) {
        pois_mean<T>(d, P, nm, reinterpret_cast<double*>(pllc_smem), s * LPB + q, LPB * PC);
        return;
    }
    const int n = d.nx;
    const int l = blockIdx.x * LPB + q;
    const bool live = l < nm && l > 0;
    const int x0 = s * PM, nv = min(PM, n - x0);
    T* p = P + (live ? l : 0) + (long)x0 * nm;
    PChunk<T> ch;
    if (live) {
        const int jy = l / d.nz, kz = l - jy * d.nz;
        const T h = T(1.0) / (T(d.dx) * T(d.dx));
        const T bm = T(-2.0) * h + lam_y[jy] + lam_z[kz];
        const int tl = x0 + PM >= n ? nv - 1 : PM;
        T sv[PM];
        if (nv == PM) {
#pragma unroll
            for (int t = 0; t < PM; t++) sv[t] = p[(long)t * nm];
        } else {
            // past the line's end: its last row again, which no row reads
            const unsigned mi = (unsigned)nm, lim = (nv - 1) * mi;
#pragma unroll
            for (int t = 0; t < PM; t++) sv[t] = p[min(t * mi, lim)];
        }
        // row t: h x_{t-1} + bm x_t + h x_{t+1} = sv[t], Neumann ends
#pragma unroll
        for (int t = 0; t < PM; t++) {
            const T b = t == 0 && s == 0 ? bm + h : bm;
            ch.fwd(t, t == 0 && s == 0 ? T(0.0) : h, t == tl ? b + h : b, t == tl ? T(0.0) : h, sv[t]);
            row_done();
        }
        ch.fold();
    }
    chunk_couple<T>(reinterpret_cast<T*>(pllc_smem), PC, LPB, q, s, live, ch);
    if (!live) return;
    p = P + renew((long)l + (long)x0 * nm);
    if (nv == PM) {
#pragma unroll
        for (int t = 0; t < PM; t++) p[(long)t * nm] = ch.D[t];
    } else {
#pragma unroll
        for (int t = 0; t < PM; t++)
            if (t < nv) p[(long)t * nm] = ch.D[t];
    }
}

#ifdef PLLC_F64_TU
PLLC_INST(double)
#else
PLLC_INST(float)
#endif

}  // namespace pllc

// ======================================================= launch layer ====

namespace pllc {

#ifdef PLLC_F64_TU
const char* kernel_class_names =
    "stale;rhs_c;rhs_u;rhs_v;rhs_w;rhs_uvw;rhs_cuvw;sweep_y;sweep_z;sweep_x;visc;velo_ghost;div;dct;pois_x;"
    "phi_ghost;velo_corr;flux;pg;corr_pg;cfl;bulk;copy";
#endif

// launch `expr` inside the timing hook of kernel class `name`
#define PLLC_L(c, name, expr)                                \
    do {                                                     \
        if ((c).hook) (c).hook((c).hook_user, name, 0);      \
        expr;                                                \
        if ((c).hook) (c).hook((c).hook_user, name, 1);      \
    } while (0)

// blocks of kernel f (nthreads threads, sm bytes of LDS) resident on the
// device at once: the occupancy per CU times the CUs (cached per kernel
// and shape, behind a lock: handles may launch from several host threads)
template <typename K>
static int resident_blocks(K f, int nthreads, size_t sm)
{
    static std::map<std::tuple<const void*, int, size_t>, int> cache;
    static int cus = 0;
    static std::mutex mu;
    std::lock_guard<std::mutex> lk(mu);
    const auto key = std::make_tuple((const void*)f, nthreads, sm);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    if (cus == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
    }
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, nthreads, sm) != hipSuccess || per_cu <= 0)
        return 4 * cus;   // not cached: asked again next time
    cache[key] = per_cu * cus;
    return per_cu * cus;
}

// explicit stencils in reference arithmetic (IEEE quotients, the bits of the
// reference's WENO) with the Thomas line solver, else the FAST forms
template <typename T>
static inline bool fast_stencils(const Ctx<T>& c) { return c.line_solver == 0; }

// launchers without a batched form: false (and the error set) when the
// context launches over a batch
template <typename T>
static bool single(const Ctx<T>& c, const char* what)
{
    if (c.bt.nm == 1) return true;
    pllc_set_error(what, "no batched form of this operator");
    return false;
}

// Tiles of one i-plane of at most 256 threads (k, j), k from 1: a row is cut
// into as few equal parts of at most 128 points as it needs, each rounded up
// to 16 lanes (an aligned piece of a pitched row), and a tile takes as many rows as
// fit, kp points a lane (128 x 2 measured faster than 64 x 4, 32 x 8 and 256 x 1 for the cell
// kernels at 128-point rows; at 96 points 96 x 2 leaves no lane idle where
// 128 x 2 left a quarter)
static inline dim3 cell_grid(const Rng& R, dim3& blk, int kp = 1)
{
    const int nk = (R.ke + kp - 1) / kp, nt = (nk + 127) / 128, q = 16 / kp, bx = ((nk + nt - 1) / nt + q - 1) / q * q, by = 256 / bx;
    blk = dim3(bx, by, 1);
    return dim3(nt, (R.je - R.js + 1 + by - 1) / by, R.ie - R.is + 1);
}
static inline dim3 line_grid(long n) { return dim3((unsigned)((n + 255) / 256)); }
// a cell grid (planes along z) over the context's batch: nm times the planes
template <typename T>
static inline dim3 bgrid(dim3 g, const Ctx<T>& c)
{
    g.z *= (unsigned)c.bt.nm;
    return g;
}
// vector units of the device (4 in each CU)
static int simds()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    return 4 * cus;
}

// a cell grid for n fields whose threads take np consecutive planes each
template <typename T>
static inline dim3 march_grid(const Rng& R, dim3& blk, const Ctx<T>& c, int n, int& np)
{
    dim3 g = cell_grid(R, blk, KP<T>::value);
    const double waves = (double)n * c.bt.nm * c.d.nx * c.d.ny * c.d.nz / (64 * KP<T>::value) / simds();
    np = march_planes(waves, (int)g.z, n * c.bt.nm);
    g.z = (g.z + np - 1) / np * n;
    return bgrid(g, c);
}
static inline int bulk_grid(long n) { long b = (n + 255) / 256; return (int)(b > 4096 ? 4096 : (b < 1 ? 1 : b)); }

template <typename T>
static Visc4<T> muo(Ctx<T>& c) { return {c.f[MUO_CELL], c.f[MUO_XY], c.f[MUO_XZ], c.f[MUO_YZ]}; }
template <typename T>
static Visc4<T> mun(Ctx<T>& c) { return {c.f[MUN_CELL], c.f[MUN_XY], c.f[MUN_XZ], c.f[MUN_YZ]}; }

template <typename T>
void Ops<T>::stale(Ctx<T>& c, const T* qc, const T* qu, const T* qv, const T* qw)
{
    PLLC_L(c, "stale", (k_stale<T><<<1, 64, 0, c.st>>>(c.d, qc, qu, qv, qw, c.stale)));
}

// the LineSet of field F's sweep in direction DIR (coefficient source as in
// A_conc / A_umom / A_vmom / A_wmom, boundary rows as in bc_kind)
// the constant coefficients of field F's lines in direction DIR, as
// A_conc (1411-1440: del = 1/(Pe h^2), ca = cc = del, cb = -2 del) and
// A_umom/A_vmom/A_wmom (1453-1532: del = 2/(Re h) along the component's own
// direction, 1/(Re h) across) define them: {del, ca, cb, cc}
template <typename T>
void Ops<T>::line_consts(const Phys& ph, const Dims& d, int F, int DIR, T* k)
{
    const T h = DIR == 0 ? T(d.dx) : DIR == 1 ? T(d.dy) : T(d.dz);
    k[0] = k[1] = k[2] = k[3] = T(0);
    if (F == FC) {
        const T del = T(1.0) / (T(ph.Pe) * h * h);
        k[1] = del;
        k[3] = del;
        k[2] = (DIR == 2) ? (-del - del) : -(del + del);
    } else {
        const bool normal = (F == FU && DIR == 0) || (F == FV && DIR == 1) || (F == FW && DIR == 2);
        k[0] = (normal ? T(2.0) : T(1.0)) / (T(ph.Re) * h);
    }
}

template <typename T>
static LineSet<T> line_set(Ctx<T>& c, int F, int DIR, T* S, T* CC, const Visc4<T>& mu, const T* qold, T* qnew,
                           T* N, const T* Nm1)
{
    LineSet<T> L{};
    L.S = S; L.CC = CC; L.R = field_rng(c.d, F);
    const T h = DIR == 0 ? T(c.d.dx) : DIR == 1 ? T(c.d.dy) : T(c.d.dz);
    L.h = h;
    L.rh = DIR == 0 ? c.d.rdx : DIR == 1 ? c.d.rdy : c.d.rdz;
    T k[4];
    Ops<T>::line_consts(c.ph, c.d, F, DIR, k);
    L.del = k[0]; L.ca = k[1]; L.cb = k[2]; L.cc = k[3];
    if (F == FC) {
        L.mu = nullptr;
    } else {
        const bool normal = (F == FU && DIR == 0) || (F == FV && DIR == 1) || (F == FW && DIR == 2);
        const long off[3] = {-c.d.sx, -c.d.sy, -1};
        if (normal) { L.mu = mu.cell; L.mu_off = off[DIR]; }
        else if ((F == FU && DIR == 1) || (F == FV && DIR == 0)) L.mu = mu.xy;
        else if ((F == FU && DIR == 2) || (F == FW && DIR == 0)) L.mu = mu.xz;
        else L.mu = mu.yz;
    }
    if (DIR == 1) { L.bc0 = bc_kind(F, 0); L.bc1 = bc_kind(F, 1); }
    else if (DIR == 2) { L.bc0 = bc_kind(F, 2); L.bc1 = bc_kind(F, 3); }
    else { L.bc0 = bc_kind(F, 4); L.bc1 = 0; }
    L.qold = qold; L.qnew = qnew; L.N = N; L.Nm1 = Nm1;
    L.ghost_c = (F == FC && DIR == 0) ? 1 : 0;
    L.ghost_v = 0;
    L.F = F;
    return L;
}

// chunks per line of the partitioned solve for lines of nmin..nmax rows along
// DIR, or 0 when the lines do not allow it.  z: a chunk is a lane of a wave.  x
// (y-lines have at most 1024 rows): at least two lines of 256 chunks in a
// block; the lines' pieces of a row get short (8 bytes a chunk's lane, 7 lines
// at 1030 rows), yet 1030x33x20 FP64 takes 9.6 ms a step with one thread per
// line and 0.94 so, 4096x16x16 mixed 33.8 and 0.82.
static inline int part_chunks(int nmin, int nmax, int DIR)
{
    const int P = (nmax + PM - 1) / PM;
    return nmin < 3 || P > (DIR == 2 ? 64 : 256) ? 0 : P;
}

template <typename T>
bool Ops<T>::batchable(const Ctx<T>& c)
{
    if (sizeof(T) != 4 || c.line_solver != 0 || !c.dsmall || c.cbf || c.ncorr) return false;
    if ((long)c.d.ny * c.d.nz > BULK1_MAX || part_chunks(c.d.nx, c.d.nx, 0) == 0) return false;
    for (int DIR = 0; DIR < 3; DIR++) {
        int nmin = 1 << 30, nmax = 0;
        for (int F = FC; F <= FW; F++) {
            const Rng R = field_rng(c.d, F);
            const int n = DIR == 0 ? R.ie - R.is + 1 : DIR == 1 ? R.je - R.js + 1 : R.ke - R.ks + 1;
            if (F == FC) {
                if (part_chunks(n, n, DIR) == 0) return false;
                continue;
            }
            nmin = std::min(nmin, n);
            nmax = std::max(nmax, n);
        }
        if (part_chunks(nmin, nmax, DIR) == 0) return false;
    }
    return true;
}

// y, z then x sweeps of up to three fields at once (one launch per direction)
template <typename T>
static void adi_sets(Ctx<T>& c, T g, T r, int slot, const int* F, int nset, T* const* S, T* const* CC,
                     const Visc4<T>& mu, T* const* qold, T* const* qnew, T* const* N, T* const* Nm1,
                     bool vghost = false)
{
    static const char* nm[3] = {"sweep_x", "sweep_y", "sweep_z"};
    const int order[3] = {1, 2, 0};
    for (int t = 0; t < 3; t++) {
        const int DIR = order[t];
        LineSets<T> ls{};
        long lines = 0, lanes = 0;
        for (int q = 0; q < nset; q++) {
            ls.s[q] = line_set<T>(c, F[q], DIR, S[q], CC[q], mu, qold[q], qnew[q], N[q], Nm1[q]);
            LineSet<T>& L = ls.s[q];
            if (vghost && DIR == 0 && F[q] != FC) L.ghost_v = F[q];
            L.jg = L.ghost_c || L.ghost_v == FU || L.ghost_v == FW;
            L.kg = L.ghost_c || L.ghost_v == FU || L.ghost_v == FV;
            L.inlet = L.ghost_v == FV || L.ghost_v == FW;
            const Rng& R = L.R;
            const long ni = R.ie - R.is + 1, nj = R.je - R.js + 1, nk = R.ke - R.ks + 1;
            lines = std::max(lines, DIR == 0 ? nj * nk : DIR == 1 ? ni * nk : ni * nj);
            // the partitioned x- and y-sweeps' lanes
            lanes = std::max(lanes, (DIR == 0 ? nj + 2 * L.jg : ni) * line_row(c.d.nz));
        }
        int nmax = 0, nmin = 1 << 30;
        for (int q = 0; q < nset; q++) {
            const Rng& R = ls.s[q].R;
            const int n = DIR == 0 ? R.ie - R.is + 1 : DIR == 1 ? R.je - R.js + 1 : R.ke - R.ks + 1;
            nmax = std::max(nmax, n);
            nmin = std::min(nmin, n);
        }
        const int P = c.line_solver == 0 ? part_chunks(nmin, nmax, DIR) : 0;
        if (P > 0 && DIR != 2) {
            // lines per block: y-lines 256 bytes of a row (short pieces of it
            // fetch more lines than they use);
            // x-lines, which couple more chunks, 16 lines (256x128x128, y at 16:
            // 65 us instead of 57 FP64, 41 instead of 27 FP32; x at 32: 86
            // instead of 83 FP64, 15.3 instead of 12.0 for c in FP32)
            const int most = std::max(1, PART_THREADS / P);
            int LPB = std::min(DIR == 0 ? 16 : 256 / (int)sizeof(T), most);
            if (c.lpb[DIR] > 0) LPB = std::min(c.lpb[DIR], most);   // tuned
            // block count rounded up to a multiple of 8 (XCD order); the
            // blocks past the last line do nothing
            const dim3 blk(LPB, P, 1), grd((unsigned)(((lanes + LPB - 1) / LPB + 7) / 8 * 8), nset, c.bt.nm);
            const size_t sm = (size_t)6 * P * LPB * sizeof(T);
            if (DIR == 0)
                PLLC_L(c, nm[0], (k_sweep_part<T, 0><<<grd, blk, sm, c.st>>>(c.d, ls, c.scal, slot, g, r, c.bt)));
            else
                PLLC_L(c, nm[1], (k_sweep_part<T, 1><<<grd, blk, sm, c.st>>>(c.d, ls, c.scal, slot, g, r, c.bt)));
            continue;
        }
        int nj = 0, ni = 0;
        for (int q = 0; q < nset; q++) {
            const Rng& R = ls.s[q].R;
            nj = std::max(nj, R.je - R.js + 1);
            ni = std::max(ni, R.ie - R.is + 1);
        }
        if (P > 0) {
            // z-lines: a wave takes 64 / G lines of an i-plane, G lanes each
            const int LW = z_lines_per_wave(nmax), G = 64 / LW, nbx = (nj + LW - 1) / LW, ntiles = nbx * ni * nset;
            const int nw = z_block_waves(c.lpb[2], nmax, Z_WAVES);
            const size_t sm = (size_t)nw * Z_TILE * sizeof(T);
            // a multiple of 8 blocks (XCD order); the tiles past the last do nothing
            const dim3 gz((unsigned)((ntiles + nw * 8 - 1) / (nw * 8) * 8), c.bt.nm, 1);
            PLLC_L(c, nm[2], (k_sweep_wave_z<T><<<gz, 64 * nw, sm, c.st>>>(c.d, ls, c.scal, g, r, G, nbx, ni, ntiles,
                                                                          c.bt)));
            continue;
        }
        if (!single(c, "sweep")) return;
        const dim3 grd((unsigned)((lines + 255) / 256), nset, 1);
        if (DIR == 0) PLLC_L(c, nm[0], (k_sweep<T, 0><<<grd, 256, 0, c.st>>>(c.d, ls, c.scal, slot, g, r)));
        else if (DIR == 1) PLLC_L(c, nm[1], (k_sweep<T, 1><<<grd, 256, 0, c.st>>>(c.d, ls, c.scal, slot, g, r)));
        else {
            // z-lines: one block per 64 lines of an i-plane
            const dim3 gz((nj + ZL - 1) / ZL, ni, nset);
            PLLC_L(c, nm[2], (k_sweep_z_lds<T><<<gz, ZL, 0, c.st>>>(c.d, ls, c.scal, g, r)));
        }
    }
}

// the field the explicit part of F leaves its source in.  With several
// components u's, v's and w's are F_SRC, F_SRC2 and F_SRC3, u's F_SRC4 where
// the concentration's (F_SRC) is still needed (split).
template <typename T>
static T* src_field(Ctx<T>& c, int F, bool several, bool split)
{
    if (!several || F == FC) return c.f[F_SRC];
    T* s = c.f[F == FU ? (split ? F_SRC4 : F_SRC) : F == FV ? F_SRC2 : F_SRC3];
    return s ? s : c.f[F_SRC];
}

// the explicit parts of the fields in the mask (bit 0 c, 1 u, 2 v, 3 w)
template <typename T>
static void rhs_set(Ctx<T>& c, int fields, double g, double r, const T* un, const T* vn, const T* wn, bool split)
{
    static const char* const names[16] = {"",        "rhs_c", "rhs_u", "", "rhs_v", "", "", "", "rhs_w", "",
                                          "",        "",      "",      "", "rhs_uvw", "rhs_cuvw"};
    const bool several = (fields & 14) == 14;
    RhsSets<T> rs;
    rs.n = 0;
    for (int F = FC; F <= FW; F++) {
        if (!(fields & (1 << F))) continue;
        const int b = F == FC ? C_OLD : F == FU ? U_OLD : F == FV ? V_OLD : W_OLD;
        const int n = F == FC ? C_N : b + 3;
        rs.s[rs.n++] = {F, F == FC ? nullptr : c.f[b + 2], c.f[n + 1], c.f[n], src_field(c, F, several, split)};
    }
    dim3 blk;
    int np;
    const dim3 grd = march_grid(field_rng(c.d, FC), blk, c, rs.n, np);
    auto go = [&](auto fast, auto bv) {
        PLLC_L(c, names[fields], (k_rhs<T, decltype(fast)::value, decltype(bv)::value><<<grd, blk, 0, c.st>>>(
                                     c.d, c.ph, rs, c.f[C_OLD], un, vn, wn, muo(c), c.f[C_NEW], c.ncorr, c.stale, c.scal,
                                     T(g), T(r), np, c.bt)));
    };
    const bool fast = fast_stencils(c);
    if (c.bt.nm > 1) fast ? go(std::true_type{}, std::true_type{}) : go(std::false_type{}, std::true_type{});
    else fast ? go(std::true_type{}, std::false_type{}) : go(std::false_type{}, std::false_type{});
}

template <typename T>
void Ops<T>::concentration(Ctx<T>& c, double g, double r, int slot, const T* un, const T* vn, const T* wn)
{
    rhs_set<T>(c, 1, g, r, un, vn, wn, false);
    concentration_implicit(c, g, r, slot);
}

template <typename T>
void Ops<T>::concentration_implicit(Ctx<T>& c, double g, double r, int slot)
{
    const int F[1] = {FC};
    T* S[1] = {c.f[F_SRC]};
    T* CC[1] = {c.f[F_CC]};
    T* qo[1] = {c.f[C_OLD]};
    T* qn[1] = {c.f[C_NEW]};
    T* N[1] = {c.f[C_N]};
    T* Nm[1] = {c.f[C_NM1]};
    adi_sets<T>(c, T(g), T(r), slot, F, 1, S, CC, Visc4<T>{nullptr, nullptr, nullptr, nullptr}, qo, qn, N, Nm);
}

template <typename T>
void Ops<T>::viscosity(Ctx<T>& c, const T* cn, T* const mu[4])
{
    // chunks of 256 lanes per (j, k) plane, rounded up to a multiple of 8
    const int nb = (int)(((long)(c.d.ny + 2) * (c.d.nz + 2) + 256 * 8 - 1) / (256 * 8)) * 8;
    const dim3 grd(nb, c.d.nx + 2, c.bt.nm);
    if (c.bt.nm > 1)
        PLLC_L(c, "visc", (k_visc<T, true><<<grd, 256, 0, c.st>>>(c.d, c.ph, cn, mu[0], mu[1], mu[2], mu[3], c.bt)));
    else
        PLLC_L(c, "visc", (k_visc<T><<<grd, 256, 0, c.st>>>(c.d, c.ph, cn, mu[0], mu[1], mu[2], mu[3], c.bt)));
}

// the sweeps of the components in the mask (bit 0 u, 1 v, 2 w) from the
// sources of their explicit parts.  With several components the sweeps of
// all of them share launches; the components are independent (each reads
// only old velocities, c_new and the viscosities), so this equals xmom; ymom;
// zmom (179-181).
template <typename T>
static void momentum_sweeps(Ctx<T>& c, int comps, double gd, double rd, int slot, bool vghost, bool split)
{
    const bool several = comps == 7;
    int F[3], n = 0;
    T *S[3], *CC[3], *qo[3], *qn[3], *N[3], *Nm[3];
    const int ccs[3] = {F_CC, F_CC2, F_CC3};
    for (int q = 0; q < 3; q++) {
        if (!(comps & (1 << q))) continue;
        const int b = q == 0 ? U_OLD : q == 1 ? V_OLD : W_OLD;
        F[n] = FU + q; S[n] = src_field(c, FU + q, several, split);
        CC[n] = c.f[ccs[n]] ? c.f[ccs[n]] : c.f[F_CC];
        qo[n] = c.f[b]; qn[n] = c.f[b + 1]; N[n] = c.f[b + 3]; Nm[n] = c.f[b + 4];
        n++;
    }
    adi_sets<T>(c, T(gd), T(rd), slot, F, n, S, CC, mun(c), qo, qn, N, Nm, vghost);
}

template <typename T>
void Ops<T>::momentum(Ctx<T>& c, int comp, double g, double r, int slot)
{
    rhs_set<T>(c, 2 << comp, g, r, c.f[U_OLD], c.f[V_OLD], c.f[W_OLD], false);
    momentum_sweeps<T>(c, 1 << comp, g, r, slot, false, false);
}

template <typename T>
void Ops<T>::momentum3(Ctx<T>& c, double g, double r, int slot, bool ghosts)
{
    rhs_set<T>(c, 14, g, r, c.f[U_OLD], c.f[V_OLD], c.f[W_OLD], false);
    momentum_sweeps<T>(c, 7, g, r, slot, ghosts, false);
}

template <typename T>
void Ops<T>::explicit_parts(Ctx<T>& c, double g, double r)
{
    rhs_set<T>(c, 15, g, r, c.f[U_OLD], c.f[V_OLD], c.f[W_OLD], true);
}

template <typename T>
void Ops<T>::momentum3_implicit(Ctx<T>& c, double g, double r, int slot, bool ghosts)
{
    momentum_sweeps<T>(c, 7, g, r, slot, ghosts, true);
}

template <typename T>
void Ops<T>::velo_ghost(Ctx<T>& c)
{
    const long n = (long)c.d.nx * c.d.ny + (long)c.d.nx * c.d.nz + (long)c.d.ny * c.d.nz;
    PLLC_L(c, "velo_ghost", (k_velo_ghost<T><<<line_grid(n), 256, 0, c.st>>>(c.d, c.f[U_NEW], c.f[V_NEW], c.f[W_NEW])));
}

template <typename T>
void Ops<T>::divergence(Ctx<T>& c, double g, double r, bool write_div, bool pack)
{
    if (!single(c, "divergence")) return;
    dim3 blk;
    const dim3 grd = cell_grid(field_rng(c.d, FC), blk);
    PLLC_L(c, "div", (k_div<T><<<grd, blk, 0, c.st>>>(c.d, c.ph, c.f[U_NEW], c.f[V_NEW], c.f[W_NEW],
                                                       write_div ? c.f[DIV] : nullptr, pack ? c.P : nullptr, c.scal,
                                                       T(g), T(r))));
}

// opts kernel f in to sm bytes of dynamic LDS per block; false when the
// device cannot give them.  The limit belongs to the kernel, not to a handle,
// so it is set to what the largest of the kernel's planes takes (most; the
// device's own limit where that is less): set to sm, a handle of small planes
// lowered it under a living one of larger planes (135168 to 5120 bytes).
static bool lds_optin(const void* f, int sm, int most)
{
    int dev = 0, lim = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    if (hipDeviceGetAttribute(&lim, hipDeviceAttributeSharedMemPerBlockOptin, dev) != hipSuccess || lim <= 0)
        if (hipDeviceGetAttribute(&lim, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) return false;
    if (sm > lim) return false;
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, std::min(most, lim)) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return true;
}

template <typename T>
bool Ops<T>::dct_mfma_ready(int n)
{
    if constexpr (sizeof(T) == 4) {
        if (n != DM_N) return false;
        const int sm = DM_N * DM_P * (int)sizeof(float);
        return lds_optin((const void*)k_dct_bf16x3<false>, sm, sm) && lds_optin((const void*)k_dct_bf16x3<true>, sm, sm);
    }
    return false;
}

// the k_dct_planes form for (ny, nz): unrolled for square planes
template <typename T>
using DctPlanesFn = void (*)(int, int, int, int, T*, const T*, const T*, PhiOut<T>, DivIn<T>, Bt);
template <typename T>
static DctPlanesFn<T> dct_planes_fn(bool inv, int ny, int nz)
{
    if (ny == nz) switch (ny) {
        case 16: return inv ? k_dct_planes<T, true, 16> : k_dct_planes<T, false, 16>;
        case 32: return inv ? k_dct_planes<T, true, 32> : k_dct_planes<T, false, 32>;
        case 48: return inv ? k_dct_planes<T, true, 48> : k_dct_planes<T, false, 48>;
        case 64: return inv ? k_dct_planes<T, true, 64> : k_dct_planes<T, false, 64>;
        default: break;
        }
    return inv ? k_dct_planes<T, true, 0> : k_dct_planes<T, false, 0>;
}

// LDS of k_dct_planes: the plane, Q, Cz and Cy (one table for square planes)
template <typename T>
static int dct_planes_lds(int ny, int nz)
{
    return (2 * ny * ds_pitch(nz) + nz * ds_pitch(nz) + (ny == nz ? 0 : ny * ds_pitch(ny))) * (int)sizeof(T);
}

template <typename T>
bool Ops<T>::dct_small_ready(int ny, int nz)
{
    if (ny % 16 || nz % 16 || ny > DS_MAX || nz > DS_MAX) return false;
    const int smp = dct_planes_lds<T>(ny, nz);
    // the unrolled forms have one size each; the other one's planes take
    // less than four tables of the largest side
    const int most = ny == nz ? smp : 4 * DS_MAX * ds_pitch(DS_MAX) * (int)sizeof(T);
    return lds_optin((const void*)dct_planes_fn<T>(false, ny, nz), smp, most) &&
           lds_optin((const void*)dct_planes_fn<T>(true, ny, nz), smp, most);
}

template <typename T>
static int dct_wide_lds(int ny, int nz)
{
    return 16 * dw_tiles(ny) * dw_pitch(nz) * (int)sizeof(T);
}

template <typename T>
bool Ops<T>::dct_wide_ready(int ny, int nz)
{
    if (ny > DW_MAX || nz > DW_MAX) return false;
    const int sm = dct_wide_lds<T>(ny, nz), most = dct_wide_lds<T>(DW_MAX, DW_MAX);
    return lds_optin((const void*)k_dct_wide<T, false>, sm, most) &&
           lds_optin((const void*)k_dct_wide<T, true>, sm, most);
}

template <typename T>
bool Ops<T>::dct_fast_ready(int n)
{
    if (n == FD_N) {
        const int sm = FD_N * FD_P * (int)sizeof(T);
        return lds_optin((const void*)k_dct_plane<T, false>, sm, sm) &&
               lds_optin((const void*)k_dct_plane<T, true>, sm, sm);
    }
    if (n == 256) {
        constexpr int FL = fl_lines<T>();
        const int sm = FL * (256 + 1) * (int)sizeof(T);
        return lds_optin((const void*)k_dct_lines<T, false, 256, 1, FL>, sm, sm) &&
               lds_optin((const void*)k_dct_lines<T, false, 256, 2, FL>, sm, sm) &&
               lds_optin((const void*)k_dct_lines<T, true, 256, 1, FL>, sm, sm) &&
               lds_optin((const void*)k_dct_lines<T, true, 256, 2, FL>, sm, sm);
    }
    return false;
}

template <typename T>
void Ops<T>::dct2(Ctx<T>& c, T* io, bool inverse, T* phi, bool ghosts, const DivIn<T>* div)
{
    const DivIn<T> dv = div ? *div : DivIn<T>{};
    const int nx = c.d.nx, ny = c.d.ny, nz = c.d.nz;
    if constexpr (sizeof(T) == 4) {
        if (c.cbf && ny == DM_N && nz == DM_N) {
            // 128 x 128 FP32 planes: BF16x3 contractions on the matrix cores
            const size_t sm = (size_t)DM_N * DM_P * sizeof(float);
            if (inverse) {
                const PhiOut<float> po{phi, c.d.sx, c.d.sy, nx, ny, nz, ghosts ? 1 : 0};
                PLLC_L(c, "dct", (k_dct_bf16x3<true><<<nx, 512, sm, c.st>>>(io, io, c.cbf, po)));
            } else {
                PLLC_L(c, "dct", (k_dct_bf16x3<false><<<nx, 512, sm, c.st>>>(io, io, c.cbf, PhiOut<float>{})));
            }
            return;
        }
    }
    if (c.tw && ny == FD_N && nz == FD_N) {
        // 128 x 128 planes: the fast transform, one block per x-plane
        const size_t sm = (size_t)FD_N * FD_P * sizeof(T);
        const PhiOut<T> po{phi, c.d.sx, c.d.sy, nx, ny, nz, ghosts ? 1 : 0};
        if (inverse)
            PLLC_L(c, "dct", (k_dct_plane<T, true><<<nx, FdCfg<T>::threads, sm, c.st>>>(io, io, c.tw, po, dv)));
        else
            PLLC_L(c, "dct", (k_dct_plane<T, false><<<nx, FdCfg<T>::threads, sm, c.st>>>(io, io, c.tw,
                                                                                           PhiOut<T>{}, dv)));
        return;
    }
    if (c.tw && ny == 256 && nz == 256) {
        // 256 x 256 planes: the fast transform in two launches of FL lines
        // per block, rows (z) then columns (y); the inverse's rows write phi
        constexpr int N = 256, FL = fl_lines<T>();
        const size_t sm = (size_t)FL * (N + 1) * sizeof(T);
        const unsigned nb = (unsigned)((long)nx * N / FL);
        if (!inverse) {
            PLLC_L(c, "dct", (k_dct_lines<T, false, N, 2, FL><<<nb, 8 * FL, sm, c.st>>>(io, io, c.tw, PhiOut<T>{}, dv)));
            PLLC_L(c, "dct", (k_dct_lines<T, false, N, 1, FL><<<nb, 8 * FL, sm, c.st>>>(io, io, c.tw, PhiOut<T>{},
                                                                                          DivIn<T>{})));
        } else {
            const PhiOut<T> po{phi, c.d.sx, c.d.sy, nx, ny, nz, ghosts ? 1 : 0};
            PLLC_L(c, "dct", (k_dct_lines<T, true, N, 1, FL><<<nb, 8 * FL, sm, c.st>>>(io, io, c.tw, PhiOut<T>{},
                                                                                         DivIn<T>{})));
            PLLC_L(c, "dct", (k_dct_lines<T, true, N, 2, FL><<<nb, 8 * FL, sm, c.st>>>(io, io, c.tw, po, DivIn<T>{})));
        }
        return;
    }
    if (c.dsmall) {
        // small planes: both contractions in one launch, persistent blocks
        // over the planes (of every member of a batch)
        const size_t sm = (size_t)dct_planes_lds<T>(ny, nz);
        const int np = nx * c.bt.nm;
        const PhiOut<T> po{inverse ? phi : nullptr, c.d.sx, c.d.sy, nx, ny, nz, ghosts ? 1 : 0};
        const T* tz = inverse ? c.Ciz : c.Cfz;
        const T* ty = inverse ? c.Ciy : c.Cfy;
        const DctPlanesFn<T> kern = dct_planes_fn<T>(inverse, ny, nz);
        const int nthr = dct_planes_threads(ny == nz ? ny : 0);
        const int G = std::max(1, std::min(np, resident_blocks(kern, nthr, sm)));
        PLLC_L(c, "dct", (kern<<<G, nthr, sm, c.st>>>(ny, nz, nx, np, io, tz, ty, po, dv, c.bt)));
        return;
    }
    if (!single(c, "dct2")) return;
    if (c.Ofz) {
        const size_t sm = (size_t)dct_wide_lds<T>(ny, nz);
        const int nthr = 64 * dw_waves(ny, nz);
        const PhiOut<T> po{inverse ? phi : nullptr, c.d.sx, c.d.sy, nx, ny, nz, ghosts ? 1 : 0};
        if (inverse)
            PLLC_L(c, "dct", (k_dct_wide<T, true><<<nx, nthr, sm, c.st>>>(ny, nz, io, c.Oiz, c.Oiy, po, dv)));
        else
            PLLC_L(c, "dct", (k_dct_wide<T, false><<<nx, nthr, sm, c.st>>>(ny, nz, io, c.Ofz, c.Ofy, po, dv)));
        return;
    }
    const long R = (long)nx * ny, plane = (long)ny * nz;
    const dim3 gz((nz + 127) / 128, (unsigned)((R + 63) / 64), 1), gy((nz + 127) / 128, (ny + 63) / 64, nx);
    if (!inverse) {
        // z: Q[r][kz] = sum_m io[r][m] Cfz[kz][m]; then y: io[x] = Cfy Q[x]
        PLLC_L(c, "dct", (k_gemm<T, true><<<gz, 256, 0, c.st>>>((int)R, nz, nz, io, 0, c.Cfz, 0, c.Q, 0,
                                                                  PhiOut<T>{})));
        PLLC_L(c, "dct", (k_gemm<T, false><<<gy, 256, 0, c.st>>>(ny, nz, ny, c.Cfy, 0, c.Q, plane, io, plane,
                                                                   PhiOut<T>{})));
    } else {
        // z then y, as the forward transform; with phi set the y pass writes
        // phi (and with ghosts its face ghosts) instead of io
        PLLC_L(c, "dct", (k_gemm<T, true><<<gz, 256, 0, c.st>>>((int)R, nz, nz, io, 0, c.Ciz, 0, c.Q, 0,
                                                                  PhiOut<T>{})));
        const PhiOut<T> po{phi, c.d.sx, c.d.sy, nx, ny, nz, ghosts ? 1 : 0};
        PLLC_L(c, "dct", (k_gemm<T, false><<<gy, 256, 0, c.st>>>(ny, nz, ny, c.Ciy, 0, c.Q, plane, io, plane, po)));
    }
}

template <typename T>
void Ops<T>::poisson(Ctx<T>& c, double g, double r, bool from_div, bool ghosts, bool from_velo)
{
    dim3 blk;
    const dim3 grd = cell_grid(field_rng(c.d, FC), blk);
    const long nm = (long)c.d.ny * c.d.nz;
    if (from_div) {
        if (!single(c, "poisson")) return;
        PLLC_L(c, "div", (k_pack_div<T><<<grd, blk, 0, c.st>>>(c.d, c.ph, c.f[DIV], c.P, c.scal, T(g), T(r))));
    }
    // the right-hand side made in the forward transform's load, or packed
    // first for the transforms without one (k_gemm, k_dct_bf16x3).  (A batch's
    // blocks take many planes in turn; packed first its 64 members measured
    // 8.94 ms a step, this 8.91.)
    DivIn<T> dv{};
    if (from_velo) {
        if (!c.cbf && (c.tw || c.dsmall || c.Ofz))
            dv = {c.f[U_NEW], c.f[V_NEW], c.f[W_NEW], c.scal, c.d, c.ph.Re, T(T(g) + T(r))};
        else divergence(c, g, r, false, true);
    }
    // the spectrum, in place in P
    T* sp = c.P;
    dct2(c, sp, false, nullptr, false, &dv);
    const int PC = c.line_solver == 0 ? part_chunks(c.d.nx, c.d.nx, 0) : 0;
    if (PC > 0) {
        // 128 bytes of a row per block, more where that is less than 256
        // threads (512x256x256: 64 bytes 134 us FP64, 128 bytes 86; mixed 32
        // bytes 138 us, 64 bytes 68, 128 bytes 57)
        const int LPB = std::min(std::min(64, POIS_THREADS / PC), std::max((int)(128 / sizeof(T)), 256 / PC));
        const size_t sm = sizeof(T) * 6 * PC * LPB;
        // the last block is the mean line's
        const dim3 gp((unsigned)((nm + LPB - 1) / LPB) + 1, c.bt.nm, 1);
        PLLC_L(c, "pois_x", (k_pois_part<T><<<gp, dim3(LPB, PC, 1), sm, c.st>>>(c.d, c.lam_y, c.lam_z, sp, c.bt)));
    } else {
        if (!single(c, "poisson")) return;
        PLLC_L(c, "pois_x", (k_pois_x<T><<<line_grid(nm), 256, 0, c.st>>>(c.d, c.lam_y, c.lam_z, sp, c.QC, c.lam00)));
    }
    // the inverse transform's last pass writes phi, normalised
    dct2(c, sp, true, c.f[PHI], ghosts);
}

template <typename T>
void Ops<T>::phi_ghost(Ctx<T>& c)
{
    const long n = (long)c.d.nx * c.d.ny + (long)c.d.nx * c.d.nz + (long)c.d.ny * c.d.nz;
    PLLC_L(c, "phi_ghost", (k_phi_ghost<T><<<line_grid(n), 256, 0, c.st>>>(c.d, c.f[PHI])));
}

template <typename T>
void Ops<T>::velo_correction(Ctx<T>& c, double g, double r, int slot)
{
    dim3 blk;
    const dim3 grd = cell_grid(field_rng(c.d, FC), blk);
    if (!single(c, "velo_correction")) return;
    PLLC_L(c, "velo_corr", (k_velo_corr<T><<<grd, blk, 0, c.st>>>(c.d, c.ph, c.f[PHI], c.f[U_NEW], c.f[V_NEW],
                                                                   c.f[W_NEW], c.scal, T(g), T(r))));
    PLLC_L(c, "flux", (k_flux_rows<T><<<c.d.ny, 64, 0, c.st>>>(c.d, c.f[U_NEW], c.part, c.bt)));
    PLLC_L(c, "flux", (k_flux_apply<T><<<c.d.ny, 128, 0, c.st>>>(c.d, c.ph, c.f[U_NEW], c.scal, c.part, slot, c.bt)));
}

template <typename T>
bool Ops<T>::correction_and_gradient(Ctx<T>& c, double g, double r, int slot, bool ghosts, int next, double alpha)
{
    // the form with several points a thread from 4 of its one-plane waves per
    // vector unit on (measured at k_corr_pg_run; 64x32x32 has 0.5 in FP64,
    // 128x64x64 4, 600x20x20 3.7 (8.2 us, several points 9.4) and 150x70x51 8
    // in FP32)
    dim3 blk;
    dim3 grd = cell_grid(field_rng(c.d, FC), blk, KP<T>::value);
    const bool run = (double)c.bt.nm * c.d.nx * c.d.ny * c.d.nz / (64 * KP<T>::value) >= 4.0 * simds();
    if (run) grd.z = (grd.z + CORR_PLANES - 1) / CORR_PLANES;
    else grd = cell_grid(field_rng(c.d, FC), blk);
    grd = bgrid(grd, c);
    const dim3 gf(c.d.ny, c.bt.nm, 1);
    const bool small = c.d.ny <= FE_MAX && c.d.nz <= FE_MAX;
    auto go = [&](auto bv) {
        constexpr bool B = decltype(bv)::value;
        auto* k = run ? k_corr_pg_run<T, B> : k_corr_pg<T, B>;
        PLLC_L(c, "corr_pg", (k<<<grd, blk, 0, c.st>>>(c.d, c.ph, mun(c), c.f[PHI], c.f[U_NEW], c.f[V_NEW],
                                                       c.f[W_NEW], c.f[U_PG], c.f[V_PG], c.f[W_PG], c.scal, T(g), T(r),
                                                       ghosts ? 1 : 0, c.bt)));
        if (small) {
            PLLC_L(c, "flux", (k_step_end<T, B><<<dim3(next < 0 ? 1 : 2, c.bt.nm), 1024, 0, c.st>>>(
                                  c.d, c.ph, c.f[U_NEW], c.scal, slot, next, alpha, c.tval, c.f[C_NEW], c.f[V_NEW],
                                  c.f[W_NEW], c.stale, c.bt)));
            return;
        }
        PLLC_L(c, "flux", (k_flux_rows<T><<<gf, 64, 0, c.st>>>(c.d, c.f[U_NEW], c.part, c.bt)));
        PLLC_L(c, "flux", (k_flux_apply<T, B><<<gf, 128, 0, c.st>>>(c.d, c.ph, c.f[U_NEW], c.scal, c.part, slot,
                                                                     c.bt)));
    };
    if (c.bt.nm > 1) go(std::true_type{});
    else go(std::false_type{});
    return small;
}

template <typename T>
void Ops<T>::pressure_gradient(Ctx<T>& c, double g, double r, int mask)
{
    dim3 blk;
    const dim3 grd = cell_grid(field_rng(c.d, FC), blk);
    if (!single(c, "pressure_gradient")) return;
    PLLC_L(c, "pg", (k_pg<T><<<grd, blk, 0, c.st>>>(c.d, c.ph, mun(c), c.f[PHI], c.f[U_PG], c.f[V_PG], c.f[W_PG],
                                                     c.scal, T(g), T(r), mask)));
}

template <typename T>
void Ops<T>::cfl(Ctx<T>& c, bool start, double alpha)
{
    dim3 blk;
    dim3 grd = cell_grid(field_rng(c.d, FC), blk);
    grd.z = (c.d.nx + CFL_PLANES - 1) / CFL_PLANES;
    const bool with = start && (long)c.d.ny * c.d.nz <= BULK1_MAX;
    // partials of member m at m * bt.np (one per block)
    PLLC_L(c, "cfl", (k_cfl_partial<T><<<bgrid(grd, c), blk, 0, c.st>>>(c.d, c.f[U_OLD], c.f[V_OLD], c.f[W_OLD],
                                                                        c.part, c.bt)));
    PLLC_L(c, "cfl", (k_cfl_final<T><<<dim3(c.bt.nm, with ? 3 : 1), 1024, 0, c.st>>>(
                         c.part, (long)grd.x * grd.y * grd.z, c.ph.CFLmax, c.ph.Timestep, c.scal, c.d, alpha,
                         with ? c.tval : nullptr, c.f[C_OLD], c.f[U_OLD], c.f[V_OLD], c.f[W_OLD], c.stale, c.bt)));
    if (start && !with) bulk_stale(c, 0, alpha, true, c.f[C_OLD], c.f[U_OLD], c.f[V_OLD], c.f[W_OLD]);
}

template <typename T>
void Ops<T>::bulk(Ctx<T>& c, int slot, double alpha, bool advance_t)
{
    const long np = (long)c.d.ny * c.d.nz;
    if (np <= BULK1_MAX) {
        PLLC_L(c, "bulk", (k_bulk_stale<T><<<dim3(1, c.bt.nm), 1024, 0, c.st>>>(c.d, c.f[U_OLD], c.scal, slot, alpha,
                                                                              advance_t ? c.tval : nullptr, nullptr,
                                                                              nullptr, nullptr, nullptr, nullptr,
                                                                              c.bt)));
        return;
    }
    if (!single(c, "bulk")) return;
    const int nb = (int)((np + 255) / 256);
    PLLC_L(c, "bulk", (k_bulk_partial<T><<<nb, 256, 0, c.st>>>(c.d, c.f[U_OLD], c.part)));
    PLLC_L(c, "bulk", (k_bulk_final<T><<<1, 256, 0, c.st>>>(c.part, nb, c.scal, slot, alpha,
                                                          advance_t ? c.tval : nullptr)));
}

template <typename T>
void Ops<T>::bulk_stale(Ctx<T>& c, int slot, double alpha, bool advance_t, const T* qc, const T* qu, const T* qv,
                        const T* qw)
{
    if ((long)c.d.ny * c.d.nz > BULK1_MAX) {
        if (!single(c, "bulk_stale")) return;
        bulk(c, slot, alpha, advance_t);
        stale(c, qc, qu, qv, qw);
        return;
    }
    PLLC_L(c, "bulk", (k_bulk_stale<T><<<dim3(2, c.bt.nm), 1024, 0, c.st>>>(c.d, c.f[U_OLD], c.scal, slot, alpha,
                                                                          advance_t ? c.tval : nullptr, qc, qu, qv,
                                                                          qw, c.stale, c.bt)));
}

static inline int row_grid(long rows) { return (int)std::min((rows + 3) / 4, 8192L); }

template <typename T>
void Ops<T>::copy_pairs(Ctx<T>& c, const int (&pairs)[12][2], bool back)
{
    const long rows = (long)c.d.NX * c.d.NY;
    CopyPairs<T> cp;
    for (int q = 0; q < 12; q++) { cp.a[q] = c.f[pairs[q][back]]; cp.b[q] = c.f[pairs[q][!back]]; }
    PLLC_L(c, "copy", (k_copy_pairs<T><<<dim3(row_grid(rows), 12), dim3(64, 4), 0, c.st>>>(c.d, cp, rows)));
}

template <typename T>
void Ops<T>::pack(Ctx<T>& c, const T* a, double* b, long rows)
{
    k_pack<T><<<row_grid(rows), dim3(64, 4), 0, c.st>>>(c.d, a, b, rows);
}

template <typename T>
void Ops<T>::unpack(Ctx<T>& c, const double* a, T* b, long rows)
{
    k_unpack<T><<<row_grid(rows), dim3(64, 4), 0, c.st>>>(c.d, a, b, rows);
}

template <typename T>
void Ops<T>::set_scalar(Ctx<T>& c, int idx, double v)
{
    op_start(c, idx, v, idx, v, false);
}

template <typename T>
void Ops<T>::op_start(Ctx<T>& c, int i0, double v0, int i1, double v1, bool with_stale)
{
    k_set_scalars<T><<<1, 64, 0, c.st>>>(c.scal, i0, v0, i1, v1, c.d, c.f[C_OLD], c.f[U_OLD], c.f[V_OLD], c.f[W_OLD],
                                         with_stale ? c.stale : nullptr);
}

template <typename T>
void Ops<T>::shift_conc(Ctx<T>& c, T* q, const double* x, const double* shift)
{
    const long nl = (long)c.d.NY * c.d.NZ;
    k_spline_lines<T><<<(unsigned)((nl + 127) / 128), 128, 0, c.st>>>(c.d.NX, nl, c.d.NZ, c.d.sy, 1, c.d.sx, T(c.d.dx),
                                                                      x, nullptr, shift, q, c.f[F_CC], c.f[F_SRC]);
}

#ifdef PLLC_F64_TU
template struct Ops<double>;
#else
template struct Ops<float>;
#endif

#ifdef PLLC_F64_TU
void spline_line(int N, double delta, const double* x, const double* xx, double* y, double* cp, double* fp,
                 hipStream_t st)
{
    k_spline_lines<double><<<1, 64, 0, st>>>(N, 1, 1, 0, 0, 1, delta, x, xx, nullptr, y, cp, fp);
}

void thomas_lines(int nsys, int n, long ls, long rs, const double* a, double* b, double* c, double* r, double* cc,
                  int mode, hipStream_t st)
{
    k_thomas_lines<<<(nsys + 255) / 256, 256, 0, st>>>(nsys, n, ls, rs, a, b, c, r, cc, mode);
}

void weno_batch(const double* d1, const int* kk, const int* sg, double* out, int n, hipStream_t st)
{
    k_weno_batch<<<(n + 255) / 256, 256, 0, st>>>(d1, kk, sg, out, n);
}

void gemm_nn(int M, int N, int K, const double* A, long sA, const double* B, long sB, double* C, long sC, int batch,
             hipStream_t st)
{
    k_gemm<double, false><<<dim3((N + 127) / 128, (M + 63) / 64, batch), 256, 0, st>>>(M, N, K, A, sA, B, sB, C, sC,
                                                                                         PhiOut<double>{});
}

__global__ void k_scale_div(double* __restrict__ a, long n, double div)
{
    for (long l = (long)blockIdx.x * blockDim.x + threadIdx.x; l < n; l += (long)gridDim.x * blockDim.x)
        a[l] = a[l] / div;
}

void scale(double* a, long n, double div, hipStream_t st)
{
    k_scale_div<<<bulk_grid(n), 256, 0, st>>>(a, n, div);
}

#endif  // PLLC_F64_TU

}  // namespace pllc
