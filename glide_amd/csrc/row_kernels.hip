// gfx950 kernels of the residual, its derivative, the transpose operator and the
// cached adjoint smoothing passes on whole rows (row_ops.hpp): one wavefront per row segment of 64
// columns, halo lanes and rows recomputed, no intermediate in global memory.
//
// k_adjoint_rows: one cached adjoint pass in one launch.  The transpose
// operator minus the forcing for the rows of the workgroup, the cached 5x5
// patch solves, and the multipliers' update into the other of two buffers
// (neighbouring workgroups read the old ones).  MC: one colour phase of the
// red-black pass, where every facet belongs to exactly one solving cell, so the
// halo is one row above and below; otherwise the additive pass, whose facets
// also take the increments of the cells left of and above the workgroup.
// k_vjp_rows: the transpose operator alone.
// k_residual_rows, k_jvp_rows: the residual and its directional derivative.
// The tile kernels evaluated each vertex's shear for every cell and facet that
// reads it; FP64 at 1536 x 2048: residual 161 to 77 us (377 MB: 4.9 TB/s),
// derivative 240 to 84 us (453 MB: 5.4 TB/s), both the rate of a large copy.
//
// Workgroup height: a workgroup of NW wavefronts gives NW - 2 rows (MC), so 8
// wavefronts do the cell work of 1.33 rows per row and 16 of 1.14; 16 measured
// slower all the same (FP32 phase at 512 x 512 12.1 against 10.4 us, at the
// finest levels of 48 domains of 48 to 384 cells a side 69 against 62 us): a
// barrier then holds up twice the wavefronts.  Against the tile kernels (4 x 64
// cells, 512 threads, bound by VALU issue) the FP32 phase at 512 x 512 went from
// 24.8 to 10.4 us (33.0 MB of state, multipliers and the colour's factors: 3.2
// TB/s), the 48 domains' finest level from 232 to 62 us (3.8 TB/s, of 4.9 TB/s
// a large copy reaches: bound by memory), the FP64 transpose operator at 1536 x
// 2048 from 268 to 104 us (4.3 TB/s).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "row_ops.hpp"
#include "ssa_device.hpp"
#include "ssa_kernels.hpp"
#include "tab.hpp"

namespace glide {

namespace {

// Increments of a patch from its 25 cached factors (J^T d = b).
template <typename T>
__device__ __forceinline__ void solve_cached(const T A[25], const T b[5], T d[5]) {
    T y[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        T s = b[q];
#pragma unroll
        for (int k = 0; k < q; ++k) s -= A[q * 5 + k] * y[k];
        y[q] = s;
    }
#pragma unroll
    for (int q = 4; q >= 0; --q) {
        T s = y[q];
#pragma unroll
        for (int k = q + 1; k < 5; ++k) s -= A[q * 5 + k] * d[k];
        d[q] = s * A[q * 6];
    }
}

template <typename T, int NW, bool MC>
struct AdjointRows {
    static constexpr int kHaloL = MC ? 2 : 3, kHaloR = 2;
    static constexpr int kCols = kRowLanes - kHaloL - kHaloR;
    static constexpr int kAbove = MC ? 1 : 2;  // rows above the first one the workgroup updates
    static constexpr int kRows = NW - 1 - kAbove;

    // omega: the signed weight of the increments
    static __device__ __forceinline__ void pass(int bx, int by, const SsaArgs<T>& a, const T* __restrict__ cache,
                                                const T* __restrict__ lu, const T* __restrict__ lv,
                                                const T* __restrict__ lH, T* __restrict__ lu_dst,
                                                T* __restrict__ lv_dst, T* __restrict__ lH_dst,
                                                const T* __restrict__ fu, const T* __restrict__ fv,
                                                const T* __restrict__ fH, T calving_rate, T omega, int colour) {
        __shared__ typename TransposeRows<T, NW, false>::Lds s;
        const int ny = a.ny, nx = a.nx;
        const long n = (long)ny * nx;
        const int lane = threadIdx.x, w = wave_row(threadIdx.y);
        const int i = by * kRows - kAbove + w, j = bx * kCols - kHaloL + lane;
        const bool cell = i >= 0 && i < ny && j >= 0 && j < nx;
        // the wavefronts and lanes whose patches this workgroup solves
        const bool solves = cell && w > 0 && w < NW - 1 && lane >= (MC ? kHaloL : kHaloL - 1) &&
                            lane < kRowLanes - kHaloR && (!MC || ((i + j) & 1) == colour);
        // the factors are loaded ahead of the operator, whose chain hides them
        T A[25];
        if (solves) {
            const T* __restrict__ row = cache + (long)i * nx;
            const unsigned k = cache_column(j, nx, MC);
#pragma unroll
            for (int q = 0; q < 25; ++q) A[q] = (row + q * n)[k];
        }
        TransposeRows<T, NW, false> t;
        t.run(s, a, lu, lv, lH, fu, fv, fH, calving_rate, cache + (long)kAdjointCacheEta * n, w, lane, i, j);
        const T rur = lane_right(t.ru);
        T d[5] = {T(0), T(0), T(0), T(0), T(0)};
        if (solves) {
            const T b[5] = {t.ru, rur, t.rv, t.rvb, t.rH};
            solve_cached(A, b, d);
        }
        const bool own = cell && w >= kAbove && w < NW - 1 && lane >= kHaloL && lane < kRowLanes - kHaloR;
        const T lur = lane_right(t.lu), d1l = lane_left(d[1]);
        T* __restrict__ urow = lu_dst + (long)i * (nx + 1);
        T* __restrict__ vrow = lv_dst + (long)i * nx;
        if constexpr (MC) {
            // a facet is written by the cell that solves it; the domain-edge
            // facets of the other colour's cells are copied
            const bool left = lane > kHaloL && j >= 1 && j <= nx && i >= 0 && i < ny && w > 0 && w < NW - 1 &&
                              lane <= kRowLanes - kHaloR && ((i + j - 1) & 1) == colour;
            const bool act = solves;
            if (act || left) urow[j] = t.lu + omega * (act ? d[0] : d1l);
            if (act) {
                vrow[j] = t.lv + omega * d[2];
                (vrow + nx)[j] = t.lvb + omega * d[3];
            }
            if (own) {
                (lH_dst + (long)i * nx)[j] = t.lH + omega * d[4];
                if (!act) {
                    if (j == 0) urow[0] = t.lu;
                    if (j == nx - 1) urow[nx] = lur;
                    if (i == 0) vrow[j] = t.lv;
                    if (i == ny - 1) (vrow + nx)[j] = t.lvb;
                }
            }
        } else {
            // the increments of the bottom facets go to the row below
            __syncthreads();
            s.down[w][0][lane] = d[3];
            __syncthreads();
            if (own) {
                const T h = T(0.5);
                T x = h * d[0];
                if (j > 0) x += h * d1l;
                urow[j] = t.lu + omega * x;
                if (j == nx - 1) urow[nx] = lur + omega * (h * d[1]);
                x = h * d[2];
                if (i > 0) x += h * s.down[w - 1][0][lane];
                vrow[j] = t.lv + omega * x;
                if (i == ny - 1) (vrow + nx)[j] = t.lvb + omega * (h * d[3]);
                (lH_dst + (long)i * nx)[j] = t.lH + omega * d[4];
            }
        }
    }
};

template <typename T, int NW, bool MC>
__global__ __launch_bounds__(kRowLanes* NW) void k_adjoint_rows(SsaArgs<T> a, const T* __restrict__ cache,
                                                                const T* __restrict__ lu, const T* __restrict__ lv,
                                                                const T* __restrict__ lH, T* __restrict__ lu_dst,
                                                                T* __restrict__ lv_dst, T* __restrict__ lH_dst,
                                                                const T* __restrict__ fu, const T* __restrict__ fv,
                                                                const T* __restrict__ fH, T calving_rate, T omega,
                                                                int colour) {
    AdjointRows<T, NW, MC>::pass(blockIdx.x, blockIdx.y, a, cache, lu, lv, lH, lu_dst, lv_dst, lH_dst, fu, fv, fH,
                                 calving_rate, omega, colour);
}

template <typename T, int NW>
__global__ __launch_bounds__(kRowLanes* NW) void k_tab_adj_pass(const TabAdjPass<T>* __restrict__ jobs,
                                                                const int* __restrict__ start, int n, int colour) {
    const int e = tab_find(start, n, blockIdx.x);
    const TabAdjPass<T> J = jobs[e];
    const int lb = blockIdx.x - start[e];
    AdjointRows<T, NW, true>::pass(lb % J.gx, lb / J.gx, J.a, J.cache, J.lu, J.lv, J.lH, J.lu_dst, J.lv_dst, J.lH_dst,
                                   J.fu, J.fv, J.fH, J.cr, J.omega, colour);
}

// All cached additive adjoint passes of a level of at most 16 x 16 cells, in one
// workgroup: 16 lanes a row, four rows a wavefront, one wavefront per SIMD.
// Everything a pass reads besides the multipliers (stress and flux
// coefficients, forcing, the patch's 25 factors) is the same in each of them and
// stays in registers; the multipliers and the rows' exchanges are in LDS.  A pass
// is then a chain of about 200 instructions and four barriers: at 14 x 14 0.75 us
// (6.6 us in the workgroup of k_adjoint_coarse, which reads them all again).  Lanes and rows
// beyond the level compute along on clamped loads; what they hand to a
// neighbour is zero, as beyond the domain's edge.
constexpr int kTinySide = 16;
__global__ __launch_bounds__(kTinySide* kTinySide) void k_adjoint_tiny(
    SsaArgs<double> a, const double* __restrict__ cache, double* __restrict__ plu, double* __restrict__ plv,
    double* __restrict__ plH, const double* __restrict__ fu, const double* __restrict__ fv,
    const double* __restrict__ fH, double calving_rate, double omega, int n_iter) {
    using T = double;
    constexpr int N = kTinySide;
    // multipliers of the facets and cells with a frame of one, and the planes
    // handed to the row below (edH, Lyy, lH (1 - mask), d3) and above (Lxy, tA, rv)
    __shared__ T s_lu[N + 2][N + 2], s_lv[N + 2][N + 2], s_dn[4][N + 1][N], s_up[3][N + 1][N];
    const int ny = a.ny, nx = a.nx, n = ny * nx;
    const int j = threadIdx.x & (N - 1), i = threadIdx.x >> 4;
    const int ic = min(i, ny - 1), jc = min(j, nx - 1), ju = min(j, nx), iv = min(i, ny);
    const int it_ = max(ic - 1, 0), ib = min(ic + 1, ny - 1), jl = max(jc - 1, 0);
    auto U = [&](const T* p, int r, int c) { return p[r * (nx + 1) + c]; };
    auto C = [&](const T* p, int r, int c) { return p[r * nx + c]; };
    const bool cell = i < ny && j < nx, jin = j > 0 && j < nx;
    const bool vt_in = jin && i > 0 && i < ny, vb_in = jin && i + 1 < ny;
    const T D = a.dxi, hD = T(0.5) * D;

    // the state's part, once
    const T u = U(a.u, ic, ju), ur = U(a.u, ic, min(j + 1, nx)), ut = U(a.u, it_, ju), ub = U(a.u, ib, ju);
    const T v = C(a.v, iv, jc), vb = C(a.v, min(i + 1, ny), jc), vl = C(a.v, iv, jl), vbl = C(a.v, min(i + 1, ny), jl);
    const T et = vt_in ? hD * ((ut - u) + (v - vl)) : T(0), eb = vb_in ? hD * ((u - ub) + (vb - vbl)) : T(0);
    const T exx = (ur - u) * D, eyy = (v - vb) * D, qs = et * et + eb * eb;
    const T sx = T(2) * exx + eyy, sy = exx + T(2) * eyy;
    const T e2 = exx * exx + eyy * eyy + exx * eyy + T(0.25) * (qs + lane16_right(qs)) + a.P.eps_reg;
    const T* eta_c = cache + (long)kAdjointCacheEta * n;
    auto eH_at = [&](int r, int c) { return C(eta_c, r, c) * C(a.H, r, c); };
    auto g_at = [&](int r, int c) { return T(1) - (T(1) - C(a.phi, r, c)) * T(0.917); };
    auto S_at = [&](int r, int c) { return C(a.phi, r, c) * C(a.bed, r, c) + g_at(r, c) * C(a.H, r, c); };
    auto bp_at = [&](int r, int c) { return C(a.beta, r, c) * C(a.phi, r, c); };
    const T H = C(a.H, ic, jc), Hl = C(a.H, ic, jl), Ht = C(a.H, it_, jc), eta = C(eta_c, ic, jc), eH = eta * H;
    const T pe = eH * a.P.glen_p * row_rcp(e2);  // edH = pe de2
    const T eHv = T(0.25) * ((eH + eH_at(it_, jc)) + (eH_at(ic, jl) + eH_at(it_, jl)));
    const T S = S_at(ic, jc), g = g_at(ic, jc), bp = bp_at(ic, jc);
    const T dwu = -(T(0.5) * (bp_at(ic, jl) + bp) + a.P.water_drag);
    const T dwv = -(T(0.5) * (bp_at(it_, jc) + bp) + a.P.water_drag);
    T fdu, cAx, cBx, kAx, kBx, fdv, cAy, cBy, kAy, kBy;
    {
        const T sp = u * u + T(10), rs = row_rsqrt(sp), al = sp * rs, Hm = T(0.5) * (Hl + H);
        const T dS = T(0.5) * (S - S_at(ic, jl)) * D, HD = Hm * D;
        fdu = Hm - T(0.5) * (u * rs) * (H - Hl);
        cAx = T(0.5) * (u + al); cBx = T(0.5) * (u - al);
        kAx = dS - HD * g_at(ic, jl); kBx = dS + HD * g;
    }
    {
        const T sp = v * v + T(10), rs = row_rsqrt(sp), al = sp * rs, Hm = T(0.5) * (Ht + H);
        const T dS = T(0.5) * (S_at(it_, jc) - S) * D, HD = Hm * D;
        fdv = Hm - T(0.5) * (v * rs) * (Ht - H);
        cAy = T(0.5) * (v - al); cBy = T(0.5) * (v + al);
        kAy = dS + HD * g_at(it_, jc); kBy = dS - HD * g;
    }
    const T mk = C(a.mask, ic, jc), keep = T(1) - mk;
    T kH = T(1) / a.dt;
    if (calving_rate != T(0)) {
        const int jr = min(jc + 1, nx - 1);
        const T k = (T(1) - C(a.phi, ic, jc)) * ((T(1) - C(a.phi, ic, jl)) + (T(1) - C(a.phi, ic, jr)) +
                                                 (T(1) - C(a.phi, it_, jc)) + (T(1) - C(a.phi, ib, jc)));
        kH += k * calving_rate * D;
    }
    const T gu = fu ? U(fu, ic, ju) : T(0), gv = fv ? C(fv, iv, jc) : T(0), gH = fH ? C(fH, ic, jc) : T(0);
    T A[25];
#pragma unroll
    for (int q = 0; q < 25; ++q) A[q] = C(cache + (long)q * n, ic, jc);

    T lu = U(plu, ic, ju), lv = C(plv, iv, jc), lH = C(plH, ic, jc);
    const T lu_edge = U(plu, ic, nx);  // Dirichlet facets: no pass changes them
    const T lv_edge = C(plv, ny, jc);
    s_lu[i + 1][j + 1] = lu;
    s_lv[i + 1][j + 1] = lv;
    if (i == ny - 1) s_lv[ny + 1][j + 1] = lv_edge;
    if (threadIdx.x < 4 * N) s_dn[threadIdx.x >> 4][0][j] = T(0);
    if (threadIdx.x < 3 * N) s_up[threadIdx.x >> 4][N][j] = T(0);
    __syncthreads();
    const bool iin = i > 0 && i < ny;
#pragma unroll 1
    for (int it = 0; it < n_iter; ++it) {
        const T lut = s_lu[max(i, 1)][j + 1], lub = s_lu[i + 2 > N ? N : i + 2][j + 1], lvb = s_lv[i + 2][j + 1];
        const T lvl = lane16_left(lv), lvbl = lane16_left(lvb), lr = lane16_right(lu);
        const T lur = j == nx - 1 ? lu_edge : lr, lHm = lH * keep;
        const T dt_ = vt_in ? hD * ((lut - lu) + (lv - lvl)) : T(0);
        const T db = vb_in ? hD * ((lu - lub) + (lvb - lvbl)) : T(0);
        const T dxx = (lur - lu) * D, dyy = (lv - lvb) * D;
        const T ws = et * dt_ + eb * db;
        const T de2 = sx * dxx + sy * dyy + T(0.5) * (ws + lane16_right(ws));
        const T edH = pe * de2;
        const T Lxx = T(2) * (eH * (T(2) * dxx + dyy) + sx * edH), Lyy = T(2) * (eH * (dxx + T(2) * dyy) + sy * edH);
        s_dn[0][i + 1][j] = edH;
        s_dn[1][i + 1][j] = Lyy;
        s_dn[2][i + 1][j] = lHm;
        const T dx_ = (lane16_left(lHm) - lHm) * D, Lxl = lane16_left(Lxx);
        T ru = (Lxx - Lxl) * D + lu * dwu + fdu * dx_ - gu;
        const T tAx = jin ? cAx * dx_ - lu * kAx : T(0), tBx = jin ? cBx * dx_ - lu * kBx : T(0);
        __syncthreads();
        const T edHs = edH + s_dn[0][i][j], dy_ = (lHm - s_dn[2][i][j]) * D;
        const T edHl = lane16_left(edHs);
        const T Lxy = vt_in ? T(2) * (eHv * dt_ + et * (T(0.25) * (edHs + edHl))) : T(0);
        const T Lxr = lane16_right(Lxy);
        const T rv = iin ? (s_dn[1][i][j] - Lyy) * D + (Lxr - Lxy) * D + lv * dwv + fdv * dy_ - gv : T(0);
        const T tAy = iin ? cAy * dy_ - lv * kAy : T(0), tBy = iin ? cBy * dy_ - lv * kBy : T(0);
        s_up[0][i][j] = Lxy;
        s_up[1][i][j] = tAy;
        s_up[2][i][j] = rv;
        __syncthreads();
        ru += (Lxy - s_up[0][i + 1][j]) * D;
        if (!jin) ru = T(0);
        const T rr = lane16_right(ru), tAr = lane16_right(tAx);
        T rH = lHm * kH + tBx + tAr + tBy + s_up[1][i + 1][j] - T(2) * eta * de2 - gH;
        if (mk > T(0)) rH = T(0);
        const T b[5] = {ru, j == nx - 1 ? T(0) : rr, rv, s_up[2][i + 1][j], rH};
        T d[5];
        solve_cached(A, b, d);
        if (!cell) d[0] = d[1] = d[2] = d[3] = d[4] = T(0);
        s_dn[3][i + 1][j] = d[3];
        const T d1l = lane16_left(d[1]);
        lH += omega * d[4];
        lu += omega * (T(0.5) * d[0] + (j > 0 ? T(0.5) * d1l : T(0)));
        __syncthreads();
        lv += omega * (T(0.5) * d[2] + T(0.5) * s_dn[3][i][j]);
        s_lu[i + 1][j + 1] = lu;
        if (i < ny) s_lv[i + 1][j + 1] = lv;
        __syncthreads();
    }
    if (cell) {
        plu[i * (nx + 1) + j] = lu;
        plv[i * nx + j] = lv;
        plH[i * nx + j] = lH;
    }
}

constexpr int kVjpWaves = 8;
constexpr int kVjpCols = kRowLanes - 4, kVjpOutRows = kVjpWaves - 2;

// The transpose operator for the facets and cells of 60 columns and 6 rows.
template <typename T, bool DRAG>
__device__ __forceinline__ void vjp_rows(int bx, int by, const SsaArgs<T>& a, const T* __restrict__ lu,
                                         const T* __restrict__ lv, const T* __restrict__ lH,
                                         const T* __restrict__ fu, const T* __restrict__ fv,
                                         const T* __restrict__ fH, T* __restrict__ ou, T* __restrict__ ov,
                                         T* __restrict__ oH, T calving_rate, const T* __restrict__ eta_cache) {
    __shared__ typename TransposeRows<T, kVjpWaves, DRAG>::Lds s;
    const int ny = a.ny, nx = a.nx;
    const int lane = threadIdx.x, w = wave_row(threadIdx.y);
    const int i = by * kVjpOutRows - 1 + w, j = bx * kVjpCols - 2 + lane;
    TransposeRows<T, kVjpWaves, DRAG> t;
    t.run(s, a, lu, lv, lH, fu, fv, fH, calving_rate, eta_cache, w, lane, i, j);
    if (w < 1 || w > kVjpWaves - 2 || lane < 2 || lane >= kRowLanes - 2 || i > ny || j > nx) return;
    if (i < ny) (ou + (long)i * (nx + 1))[j] = t.ru;
    if (j < nx) (ov + (long)i * nx)[j] = t.rv;
    if (i < ny && j < nx) (oH + (long)i * nx)[j] = t.rH;
}

template <typename T, bool DRAG>
__global__ __launch_bounds__(kRowLanes* kVjpWaves) void k_vjp_rows(SsaArgs<T> a, const T* __restrict__ lu,
                                                                   const T* __restrict__ lv,
                                                                   const T* __restrict__ lH,
                                                                   const T* __restrict__ fu,
                                                                   const T* __restrict__ fv,
                                                                   const T* __restrict__ fH, T* __restrict__ ou,
                                                                   T* __restrict__ ov, T* __restrict__ oH,
                                                                   T calving_rate, const T* __restrict__ eta_cache) {
    vjp_rows<T, DRAG>(blockIdx.x, blockIdx.y, a, lu, lv, lH, fu, fv, fH, ou, ov, oH, calving_rate, eta_cache);
}

template <typename T>
__global__ __launch_bounds__(kRowLanes* kVjpWaves) void k_tab_vjp(const TabVjp<T>* __restrict__ jobs,
                                                                  const int* __restrict__ start, int n) {
    const int e = tab_find(start, n, blockIdx.x);
    const TabVjp<T> J = jobs[e];
    const int lb = blockIdx.x - start[e];
    vjp_rows<T, false>(lb % J.gx, lb / J.gx, J.a, J.lu, J.lv, J.lH, J.fu, J.fv, J.fH, J.ou, J.ov, J.oH, J.cr,
                       J.eta_cache);
}

// The residual with its forcing, active set and Dirichlet rows for the facets
// and cells of 60 columns and 6 rows.
template <typename T, bool DRAG>
__device__ __forceinline__ void residual_rows(int bx, int by, const SsaArgs<T>& a, T* __restrict__ ou,
                                              T* __restrict__ ov, T* __restrict__ oH, int use_forcing, int use_mask,
                                              T calving_rate) {
    using F = ForwardRows<T, kVjpWaves, DRAG, false>;
    __shared__ typename F::Lds s;
    const int ny = a.ny, nx = a.nx;
    const int lane = threadIdx.x, w = wave_row(threadIdx.y);
    const int i = by * kVjpOutRows - 1 + w, j = bx * kVjpCols - 2 + lane;
    // the rows' own values are loaded ahead of the operator, whose chain hides them
    const bool own = w >= 1 && w <= kVjpWaves - 2 && lane >= 2 && lane < kRowLanes - 2;
    const bool uf = own && i < ny && j <= nx, vf = own && i <= ny && j < nx, cf = own && i < ny && j < nx;
    const long o = (long)i * nx + j;
    T fu = T(0), fv = T(0), fH = T(0), mk = T(0), gam = T(0);
    if (use_forcing) {
        if (uf) fu = a.f_u[o + i];
        if (vf) fv = a.f_v[o];
        if (cf) fH = a.f_H[o];
    }
    if (cf) {
        mk = use_mask ? a.mask[o] : T(0);
        gam = a.gamma[o];
    }
    F t;
    t.run(s, a, nullptr, nullptr, nullptr, calving_rate, w, lane, i, j);
    if (uf) ou[o + i] = (j == 0 || j == nx) ? t.u : t.ru - fu;
    if (vf) ov[o] = (i == 0 || i == ny) ? t.v : t.rv - fv;
    if (cf) oH[o] = (T(1) - mk) * (t.rH - fH) + mk * (t.H - gam);
}

template <typename T, bool DRAG>
__global__ __launch_bounds__(kRowLanes* kVjpWaves) void k_residual_rows(SsaArgs<T> a, T* __restrict__ ou,
                                                                        T* __restrict__ ov, T* __restrict__ oH,
                                                                        int use_forcing, int use_mask,
                                                                        T calving_rate) {
    residual_rows<T, DRAG>(blockIdx.x, blockIdx.y, a, ou, ov, oH, use_forcing, use_mask, calving_rate);
}

template <typename T, bool DRAG>
__global__ __launch_bounds__(kRowLanes* kVjpWaves) void k_tab_residual(const TabResidual<T>* __restrict__ jobs,
                                                                       const int* __restrict__ start, int n) {
    const int e = tab_find(start, n, blockIdx.x);
    const TabResidual<T> J = jobs[e];
    const int lb = blockIdx.x - start[e];
    residual_rows<T, DRAG>(lb % J.gx, lb / J.gx, J.a, J.ou, J.ov, J.oH, J.use_forcing, J.use_mask, J.cr);
}

// The residual's derivative along (du, dv, dH) (glide/cuda/residuals.cu:340-660):
// Dirichlet facet rows are zero and the thickness row is (1 - mask) times the
// mass balance's derivative, as in the reference.
template <typename T, bool DRAG>
__global__ __launch_bounds__(kRowLanes* kVjpWaves) void k_jvp_rows(SsaArgs<T> a, const T* __restrict__ du,
                                                                   const T* __restrict__ dv,
                                                                   const T* __restrict__ dH, T* __restrict__ ou,
                                                                   T* __restrict__ ov, T* __restrict__ oH,
                                                                   int use_mask, T calving_rate) {
    using F = ForwardRows<T, kVjpWaves, DRAG, true>;
    __shared__ typename F::Lds s;
    const int ny = a.ny, nx = a.nx;
    const int lane = threadIdx.x, w = wave_row(threadIdx.y);
    const int i = blockIdx.y * kVjpOutRows - 1 + w, j = blockIdx.x * kVjpCols - 2 + lane;
    const bool own = w >= 1 && w <= kVjpWaves - 2 && lane >= 2 && lane < kRowLanes - 2;
    const long o = (long)i * nx + j;
    const bool cf = own && i < ny && j < nx;
    const T mk = (use_mask && cf) ? a.mask[o] : T(0);
    F t;
    t.run(s, a, du, dv, dH, calving_rate, w, lane, i, j);
    if (own && i < ny && j <= nx) ou[o + i] = (j == 0 || j == nx) ? T(0) : t.ru;
    if (own && i <= ny && j < nx) ov[o] = (i == 0 || i == ny) ? T(0) : t.rv;
    if (cf) oH[o] = (T(1) - mk) * t.rH;
}

constexpr int kAdjWaves = 8;

template <typename T, int NW, bool MC>
dim3 adjoint_grid(int ny, int nx) {
    using P = AdjointRows<T, NW, MC>;
    return dim3((nx + P::kCols - 1) / P::kCols, (ny + P::kRows - 1) / P::kRows);
}

}  // namespace

template <typename T>
hipError_t launch_adjoint_pass_fused(const SsaArgs<T>& a, const T* cache, const T* lu, const T* lv, const T* lH,
                                     T* lu_dst, T* lv_dst, T* lH_dst, const T* fu, const T* fv, const T* fH,
                                     T calving_rate, T omega, hipStream_t st) {
    if (!a.P.linear_drag) return hipErrorInvalidValue;
    TimedLaunch tl(kTimeAdjointCell, (long)a.ny * a.nx, st);
    k_adjoint_rows<T, kAdjWaves, false><<<adjoint_grid<T, kAdjWaves, false>(a.ny, a.nx), dim3(kRowLanes, kAdjWaves), 0, st>>>(
        a, cache, lu, lv, lH, lu_dst, lv_dst, lH_dst, fu, fv, fH, calving_rate, -omega, -1);
    return hipGetLastError();
}

bool adjoint_tiny_fits(const SsaArgs<double>& a) {
    return a.P.linear_drag && a.ny >= 2 && a.nx >= 2 && a.ny <= kTinySide && a.nx <= kTinySide;
}
hipError_t launch_adjoint_tiny(const SsaArgs<double>& a, const double* cache, double* lu, double* lv, double* lH,
                               const double* fu, const double* fv, const double* fH, double calving_rate,
                               double omega, int n_iter, hipStream_t st) {
    if (!adjoint_tiny_fits(a)) return hipErrorInvalidValue;
    TimedLaunch tl(kTimeAdjointCell, (long)a.ny * a.nx * n_iter, st);
    k_adjoint_tiny<<<1, kTinySide * kTinySide, 0, st>>>(a, cache, lu, lv, lH, fu, fv, fH, calving_rate, -omega, n_iter);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_adjoint_pass_mc(const SsaArgs<T>& a, const T* cache, const T* lu, const T* lv, const T* lH,
                                  T* lu_dst, T* lv_dst, T* lH_dst, const T* fu, const T* fv, const T* fH,
                                  T calving_rate, T omega, int colour, hipStream_t st) {
    if (!a.P.linear_drag) return hipErrorInvalidValue;
    TimedLaunch tl(std::is_same<T, float>::value ? kTimeAdjointMc32 : kTimeAdjointMc64, (long)a.ny * a.nx, st);
    k_adjoint_rows<T, kAdjWaves, true><<<adjoint_grid<T, kAdjWaves, true>(a.ny, a.nx), dim3(kRowLanes, kAdjWaves), 0, st>>>(
        a, cache, lu, lv, lH, lu_dst, lv_dst, lH_dst, fu, fv, fH, calving_rate, -omega, colour & 1);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_vjp(const SsaArgs<T>& a, const T* lu, const T* lv, const T* lH, const T* fu, const T* fv,
                      const T* fH, T* ou, T* ov, T* oH, T calving_rate, const T* eta_cache, hipStream_t st) {
    TimedLaunch tl(kTimeVjp, (long)a.ny * a.nx, st);
    const dim3 g((a.nx + kVjpCols) / kVjpCols, (a.ny + kVjpOutRows) / kVjpOutRows), b(kRowLanes, kVjpWaves);
    if (a.P.linear_drag)
        k_vjp_rows<T, false><<<g, b, 0, st>>>(a, lu, lv, lH, fu, fv, fH, ou, ov, oH, calving_rate, eta_cache);
    else
        k_vjp_rows<T, true><<<g, b, 0, st>>>(a, lu, lv, lH, fu, fv, fH, ou, ov, oH, calving_rate, eta_cache);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_residual(const SsaArgs<T>& a, T* ou, T* ov, T* oH, int use_forcing, int use_mask, T calving_rate,
                           hipStream_t st) {
    TimedLaunch tl(kTimeResidual, (long)a.ny * a.nx, st);
    const dim3 g((a.nx + kVjpCols) / kVjpCols, (a.ny + kVjpOutRows) / kVjpOutRows), b(kRowLanes, kVjpWaves);
    if (a.P.linear_drag)
        k_residual_rows<T, false><<<g, b, 0, st>>>(a, ou, ov, oH, use_forcing, use_mask, calving_rate);
    else
        k_residual_rows<T, true><<<g, b, 0, st>>>(a, ou, ov, oH, use_forcing, use_mask, calving_rate);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_jvp(const SsaArgs<T>& a, const T* du, const T* dv, const T* dH, T* ou, T* ov, T* oH, int use_mask,
                      T calving_rate, hipStream_t st) {
    const dim3 g((a.nx + kVjpCols) / kVjpCols, (a.ny + kVjpOutRows) / kVjpOutRows), b(kRowLanes, kVjpWaves);
    if (a.P.linear_drag)
        k_jvp_rows<T, false><<<g, b, 0, st>>>(a, du, dv, dH, ou, ov, oH, use_mask, calving_rate);
    else
        k_jvp_rows<T, true><<<g, b, 0, st>>>(a, du, dv, dH, ou, ov, oH, use_mask, calving_rate);
    return hipGetLastError();
}

// ------------------------------------------------------------ domain tables
int tab_blocks_residual(int ny, int nx, int* gx) { return tab_blocks_vjp(ny, nx, gx); }
template <typename T>
hipError_t launch_tab_residual(const TabResidual<T>* jobs, const int* start, int n, int blocks, bool linear,
                               hipStream_t st) {
    if (n <= 0 || blocks <= 0) return hipSuccess;
    if (linear) k_tab_residual<T, false><<<blocks, dim3(kRowLanes, kVjpWaves), 0, st>>>(jobs, start, n);
    else k_tab_residual<T, true><<<blocks, dim3(kRowLanes, kVjpWaves), 0, st>>>(jobs, start, n);
    return hipGetLastError();
}

int tab_blocks_adj_pass(int ny, int nx, bool fp32, int* gx) {
    const dim3 g = fp32 ? adjoint_grid<float, kAdjWaves, true>(ny, nx)
                        : adjoint_grid<double, kAdjWaves, true>(ny, nx);
    *gx = (int)g.x;
    return (int)(g.x * g.y);
}
int tab_blocks_vjp(int ny, int nx, int* gx) {
    *gx = (nx + kVjpCols) / kVjpCols;
    return *gx * ((ny + kVjpOutRows) / kVjpOutRows);
}

template <typename T>
hipError_t launch_tab_adj_pass(const TabAdjPass<T>* jobs, const int* start, int n, int blocks, int colour,
                               hipStream_t st) {
    if (n <= 0 || blocks <= 0) return hipSuccess;
    k_tab_adj_pass<T, kAdjWaves><<<blocks, dim3(kRowLanes, kAdjWaves), 0, st>>>(jobs, start, n, colour & 1);
    return hipGetLastError();
}
template <typename T>
hipError_t launch_tab_vjp(const TabVjp<T>* jobs, const int* start, int n, int blocks, hipStream_t st) {
    if (n <= 0 || blocks <= 0) return hipSuccess;
    k_tab_vjp<T><<<blocks, dim3(kRowLanes, kVjpWaves), 0, st>>>(jobs, start, n);
    return hipGetLastError();
}

#define GLIDE_ROWS_INST(T)                                                                                            \
    template hipError_t launch_adjoint_pass_fused<T>(const SsaArgs<T>&, const T*, const T*, const T*, const T*, T*,   \
                                                     T*, T*, const T*, const T*, const T*, T, T, hipStream_t);        \
    template hipError_t launch_adjoint_pass_mc<T>(const SsaArgs<T>&, const T*, const T*, const T*, const T*, T*, T*,  \
                                                  T*, const T*, const T*, const T*, T, T, int, hipStream_t);          \
    template hipError_t launch_vjp<T>(const SsaArgs<T>&, const T*, const T*, const T*, const T*, const T*, const T*,  \
                                      T*, T*, T*, T, const T*, hipStream_t);                                          \
    template hipError_t launch_residual<T>(const SsaArgs<T>&, T*, T*, T*, int, int, T, hipStream_t);                  \
    template hipError_t launch_jvp<T>(const SsaArgs<T>&, const T*, const T*, const T*, T*, T*, T*, int, T,            \
                                      hipStream_t);                                                                   \
    template hipError_t launch_tab_residual<T>(const TabResidual<T>*, const int*, int, int, bool, hipStream_t);       \
    template hipError_t launch_tab_adj_pass<T>(const TabAdjPass<T>*, const int*, int, int, int, hipStream_t);         \
    template hipError_t launch_tab_vjp<T>(const TabVjp<T>*, const int*, int, int, hipStream_t);
GLIDE_ROWS_INST(double)
GLIDE_ROWS_INST(float)
#undef GLIDE_ROWS_INST

}  // namespace glide
