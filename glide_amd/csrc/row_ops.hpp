// Building blocks of the kernels that work on whole rows of the MAC grid: a
// wavefront owns one row segment, a lane one column, and holds everything of
// its column in registers.  Neighbours in x come from the lanes beside it
// (whole-wave DPP shifts, one VALU move), neighbours in y from the wavefronts
// above and below through a few LDS planes.  Every cell, vertex and facet
// quantity is then computed once per workgroup, apart from the halo lanes and
// rows, where the tile kernels evaluated the strain invariants of a vertex four
// times and recomputed clamped 64-bit offsets for every neighbour: the
// transpose operator with the cached patch solves took 53 wave instructions
// per cell and was bound by their issue (VALU issue in 12% of wave cycles at
// eight waves per SIMD); here it takes 8 to 9.
//
// Columns outside the domain are clamped when loaded, so a lane beyond the edge
// holds the edge's value, as the reference's clamped accessors give; what is
// computed there is dropped by a select at the vertex or facet that would use it.
#pragma once

#include <hip/hip_runtime.h>

#include "ssa_device.hpp"
#include "ssa_kernels.hpp"

namespace glide {

constexpr int kRowLanes = 64;

// The value of the lane to the left / right (column j - 1 / j + 1); 0 on the
// first / last lane.  All lanes of the wavefront must be active.
__device__ __forceinline__ int dpp_left(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ int dpp_right(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x130, 0xf, 0xf, true); }
__device__ __forceinline__ float lane_left(float x) { return __int_as_float(dpp_left(__float_as_int(x))); }
__device__ __forceinline__ float lane_right(float x) { return __int_as_float(dpp_right(__float_as_int(x))); }
__device__ __forceinline__ double lane_left(double x) {
    return __hiloint2double(dpp_left(__double2hiint(x)), dpp_left(__double2loint(x)));
}
__device__ __forceinline__ double lane_right(double x) {
    return __hiloint2double(dpp_right(__double2hiint(x)), dpp_right(__double2loint(x)));
}

// The same within each row of 16 lanes.
__device__ __forceinline__ int dpp16_left(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true); }
__device__ __forceinline__ int dpp16_right(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x101, 0xf, 0xf, true); }
__device__ __forceinline__ double lane16_left(double x) {
    return __hiloint2double(dpp16_left(__double2hiint(x)), dpp16_left(__double2loint(x)));
}
__device__ __forceinline__ double lane16_right(double x) {
    return __hiloint2double(dpp16_right(__double2hiint(x)), dpp16_right(__double2loint(x)));
}

// 1/a and 1/sqrt(a) to about an ulp: the hardware estimates, refined in FP32 by
// one step as fast_rcp and fast_rsqrt refine the FP64 ones by two.  For values
// that the kernels form themselves: of an infinite argument the refinement makes
// a NaN (a caller may give an infinite step, which drops the time term).
__device__ __forceinline__ double row_rcp(double a) { return fast_rcp(a); }
__device__ __forceinline__ float row_rcp(float a) {
    const float y = __builtin_amdgcn_rcpf(a);
    return fmaf(y, fmaf(-a, y, 1.0f), y);
}
__device__ __forceinline__ double row_rsqrt(double a) { return fast_rsqrt(a); }
__device__ __forceinline__ float row_rsqrt(float a) {
    const float y = __builtin_amdgcn_rsqf(a);
    return fmaf(y, 0.5f * fmaf(-a * y, y, 1.0f), y);
}

// The row of a wavefront as a scalar, so that row pointers live in SGPRs.
__device__ __forceinline__ int wave_row(int r) { return __builtin_amdgcn_readfirstlane(r); }

// Position of cell (i, j) in a plane of the patch-factor cache.  split: the even
// columns of a row first, then the odd ones, so that the cells a colour phase
// solves in a row are contiguous.
__device__ __forceinline__ unsigned cache_column(int j, int nx, bool split) {
    return split ? (unsigned)((j >> 1) + ((j & 1) ? (nx + 1) / 2 : 0)) : (unsigned)j;
}

// Transpose operator J^T lambda - f on row segments.  A workgroup of NW
// wavefronts holds rows base .. base + NW - 1, lane l column col; the results
// are valid for wavefronts 1 .. NW - 2 (r_v also for NW - 1) and for lanes 2 ..
// 61 (r_u also for 62), i.e. the halo is two columns and one row on each side.
//
// Per cell, with exx, eyy and the vertices' shear e of the state and dxx, dyy, d
// the same of lambda, the directional derivative of the strain invariant is
//   de2 = (2 exx + eyy) dxx + (exx + 2 eyy) dyy + 0.5 sum over corners of e d,
// the viscosity's is eta p de2 / e2, and the viscosity-thickness products'
// contribution to the thickness row is -2 eta de2.
template <typename T, int NW, bool DRAG>
struct TransposeRows {
    static constexpr int kUp = DRAG ? 9 : 8;    // planes a row hands to the row below it
    static constexpr int kDown = DRAG ? 4 : 3;  // planes a row hands to the row above it
    struct Lds {
        T up[NW][kUp][kRowLanes];
        T down[NW][kDown][kRowLanes];
    };

    // this lane's multipliers (facets and cell of column j) and results
    T lu, lv, lvb, lH;
    T ru, rv, rvb, rH;
    bool masked;

    // barrier 1 and 2 of the workgroup are inside; every wavefront calls it
    __device__ __forceinline__ void run(Lds& s, const SsaArgs<T>& a, const T* __restrict__ plu,
                                        const T* __restrict__ plv, const T* __restrict__ plH,
                                        const T* __restrict__ fu, const T* __restrict__ fv,
                                        const T* __restrict__ fH, T calving_rate, const T* __restrict__ eta_cache,
                                        int w, int lane, int i, int j) {
        const int ny = a.ny, nx = a.nx;
        const T D = a.dxi;
        const int jc = clampi(j, 0, nx - 1), ju = clampi(j, 0, nx);
        const int ic = clampi(i, 0, ny - 1);
        const long rc = (long)ic * nx, rf = (long)ic * (nx + 1);
        const long rft = (long)clampi(i - 1, 0, ny - 1) * (nx + 1), rfb = (long)clampi(i + 1, 0, ny - 1) * (nx + 1);
        const long rv0 = (long)clampi(i, 0, ny) * nx, rv1 = (long)clampi(i + 1, 0, ny) * nx;
        const T u = (a.u + rf)[ju], ut = (a.u + rft)[ju], ub = (a.u + rfb)[ju];
        const T v = (a.v + rv0)[jc], vb = (a.v + rv1)[jc];
        lu = (plu + rf)[ju];
        const T lut = (plu + rft)[ju], lub = (plu + rfb)[ju];
        lv = (plv + rv0)[jc];
        lvb = (plv + rv1)[jc];
        const T H = (a.H + rc)[jc], phi = (a.phi + rc)[jc], bed = (a.bed + rc)[jc], beta = (a.beta + rc)[jc];
        const T mk = (a.mask + rc)[jc];
        lH = (plH + rc)[jc];
        const T e_in = eta_cache ? (eta_cache + rc)[jc] : (a.B + rc)[jc];
        const T gu = fu ? (fu + rf)[ju] : T(0);
        const T gv = fv ? (fv + rv0)[jc] : T(0);
        const T gH = fH ? (fH + rc)[jc] : T(0);
        masked = mk > T(0);

        const bool jin = j > 0 && j < nx;               // facet / vertex column inside the domain
        const bool vt_in = jin && i > 0 && i < ny;      // vertex (i, j)
        const bool vb_in = jin && i + 1 > 0 && i + 1 < ny;
        const T hD = T(0.5) * D;
        // shifts are taken by every lane, ahead of the selects
        const T vl = lane_left(v), vbl = lane_left(vb), lvl = lane_left(lv), lvbl = lane_left(lvb);
        const T et = vt_in ? hD * ((ut - u) + (v - vl)) : T(0);
        const T eb = vb_in ? hD * ((u - ub) + (vb - vbl)) : T(0);
        const T dt_ = vt_in ? hD * ((lut - lu) + (lv - lvl)) : T(0);
        const T db = vb_in ? hD * ((lu - lub) + (lvb - lvbl)) : T(0);
        const T ur = lane_right(u), lur = lane_right(lu);
        const T exx = (ur - u) * D, eyy = (v - vb) * D, dxx = (lur - lu) * D, dyy = (lv - lvb) * D;
        const T ws = et * dt_ + eb * db, qs = et * et + eb * eb;
        const T wsum = ws + lane_right(ws), qsum = qs + lane_right(qs);
        const T sx = T(2) * exx + eyy, sy = exx + T(2) * eyy;
        const T e2 = exx * exx + eyy * eyy + exx * eyy + T(0.25) * qsum + a.P.eps_reg;
        const T de2 = sx * dxx + sy * dyy + T(0.5) * wsum;
        const T eta = eta_cache ? e_in : T(0.5) * e_in * glen_power(e2, a.P);
        const T eH = eta * H;
        const T edH = eH * (a.P.glen_p * de2) * row_rcp(e2);
        const T Lxx = T(2) * (eH * (T(2) * dxx + dyy) + sx * edH);
        const T Lyy = T(2) * (eH * (dxx + T(2) * dyy) + sy * edH);
        const T lHm = lH * (T(1) - mk);
        const T g = T(1) - (T(1) - phi) * T(0.917);   // dS/dH
        const T S = phi * bed + g * H;                // flotation surface
        const T bp = beta * phi;

        // nonlinear drag: the facet's multiplier times the derivative of its
        // drag by a cross velocity is mu times that velocity
        T mu = T(0), dwu = -(T(0.5) * (lane_left(bp) + bp) + a.P.water_drag);
        if constexpr (DRAG) {
            const T be = T(0.5) * (lane_left(bp) + bp);
            const T z = u * u + T(0.25) * (vl * vl + v * v + vbl * vbl + vb * vb) + a.P.u_reg;
            const T pw = pow(z, a.P.drag_q), dpw = a.P.drag_q * pow(z, a.P.drag_q - T(1));
            dwu = -(be * (T(2) * dpw * u * u + pw) + a.P.water_drag);
            mu = lu * (-be * T(0.5) * dpw * u);
            if (j < 0 || j > nx || i < 0 || i >= ny) mu = T(0);
        }

        {
            T(*p)[kRowLanes] = s.up[w];
            p[0][lane] = eH; p[1][lane] = edH; p[2][lane] = Lyy; p[3][lane] = lHm;
            p[4][lane] = H; p[5][lane] = S; p[6][lane] = g; p[7][lane] = bp;
            if constexpr (DRAG) p[kUp - 1][lane] = mu;
        }

        // u facet (i, j): everything but the shear of the vertices above and below
        T tB_x, tA_x;  // what the cell right / left of the facet gets in its thickness row
        {
            const T Hl = lane_left(H), Sl = lane_left(S), gl = lane_left(g), lHl = lane_left(lHm), Lxl = lane_left(Lxx);
            const T sp = u * u + T(10), rs = row_rsqrt(sp);
            const T al = sp * rs, wa = u * rs, Hm = T(0.5) * (Hl + H);
            const T diff = (lHl - lHm) * D;
            const T fdw = Hm - T(0.5) * wa * (H - Hl);
            ru = (Lxx - Lxl) * D + lu * dwu + fdw * diff - gu;
            const T dS = T(0.5) * (S - Sl) * D, HD = Hm * D;
            tA_x = T(0.5) * diff * (u + al) - lu * (dS - HD * gl);
            tB_x = T(0.5) * diff * (u - al) - lu * (dS + HD * g);
            if (!jin) { tA_x = T(0); tB_x = T(0); }
        }
        __syncthreads();

        T Lxy = T(0), tB_y = T(0), mv = T(0);
        rv = T(0);
        if (w > 0) {
            T tA_y = T(0);
            const T(*p)[kRowLanes] = s.up[w - 1];
            const T eHt = p[0][lane], edHt = p[1][lane], Lyyt = p[2][lane], lHt = p[3][lane];
            const T Ht = p[4][lane], St = p[5][lane], gt = p[6][lane], bpt = p[7][lane];
            const T eHs = eH + eHt, edHs = edH + edHt;
            const T eHv = T(0.25) * (eHs + lane_left(eHs)), edHv = T(0.25) * (edHs + lane_left(edHs));
            if (vt_in) Lxy = T(2) * (eHv * dt_ + et * edHv);
            const T Lxyr = lane_right(Lxy);
            const T be = T(0.5) * (bpt + bp);
            T dwv = -(be + a.P.water_drag), cross = T(0);
            if constexpr (DRAG) {
                const T utr = lane_right(ut), mt = p[kUp - 1][lane];
                const T z = v * v + T(0.25) * (ut * ut + utr * utr + u * u + ur * ur) + a.P.u_reg;
                const T pw = pow(z, a.P.drag_q), dpw = a.P.drag_q * pow(z, a.P.drag_q - T(1));
                dwv = -(be * (T(2) * dpw * v * v + pw) + a.P.water_drag);
                mv = lv * (-be * T(0.5) * dpw * v);
                if (j < 0 || j >= nx || i < 0 || i > ny) mv = T(0);
                const T ms = mu + mt;
                cross = v * (ms + lane_right(ms));
            }
            const T sp = v * v + T(10), rs = row_rsqrt(sp);
            const T al = sp * rs, wa = v * rs, Hm = T(0.5) * (Ht + H);
            const T diff = (lHm - lHt) * D;
            const T fdw = Hm - T(0.5) * wa * (Ht - H);
            const T dS = T(0.5) * (St - S) * D, HD = Hm * D;
            if (i > 0 && i < ny) {
                rv = (Lyyt - Lyy) * D + (Lxyr - Lxy) * D + lv * dwv + fdw * diff - gv + cross;
                tA_y = T(0.5) * diff * (v - al) - lv * (dS + HD * gt);
                tB_y = T(0.5) * diff * (v + al) - lv * (dS - HD * g);
            }
            T(*q)[kRowLanes] = s.down[w];
            q[0][lane] = Lxy; q[1][lane] = tA_y; q[2][lane] = rv;
            if constexpr (DRAG) q[kDown - 1][lane] = mv;
        }
        __syncthreads();

        rvb = T(0);
        rH = T(0);
        if (w > 0 && w < NW - 1) {
            const T(*q)[kRowLanes] = s.down[w + 1];
            ru += (Lxy - q[0][lane]) * D;
            if constexpr (DRAG) {
                const T ms = mv + q[kDown - 1][lane];
                ru += u * (ms + lane_left(ms));
            }
            rvb = q[2][lane];
            T acc = lHm * (T(1) / a.dt) + tB_x + lane_right(tA_x) + tB_y + q[1][lane] - T(2) * eta * de2 - gH;
            if (calving_rate != T(0)) {
                const long rt = (long)clampi(ic - 1, 0, ny - 1) * nx, rb = (long)clampi(ic + 1, 0, ny - 1) * nx;
                const int jl = clampi(jc - 1, 0, nx - 1), jr = clampi(jc + 1, 0, nx - 1);
                const T k = (T(1) - phi) * ((T(1) - (a.phi + rc)[jl]) + (T(1) - (a.phi + rc)[jr]) +
                                            (T(1) - (a.phi + rt)[jc]) + (T(1) - (a.phi + rb)[jc]));
                acc += lHm * k * calving_rate * D;
            }
            if (!masked) rH = acc;
        }
        if (!jin) ru = T(0);
    }
};

// The coupled residual (JVP false) or its derivative along d = (du, dv, dH)
// (JVP true; grounded fraction, mask, bed, B and beta frozen) on row segments,
// without forcing, active set and Dirichlet rows.  Rows, lanes and halo as in
// TransposeRows: the results are valid for wavefronts 1 .. NW - 2 and lanes
// 2 .. 61.  A wavefront owns the cells, facets and top-left vertices of a row.
template <typename T, int NW, bool DRAG, bool JVP>
struct ForwardRows {
    static constexpr int kUp = JVP ? 8 : 5;  // planes a row hands to the row below it
    struct Lds {
        T up[NW][kUp][kRowLanes];
        T down[NW][2][kRowLanes];
    };

    T u, v, H, phi;    // this lane's facets and cell
    T ru, rv, rH, dH;  // dH: the direction's thickness

    // barrier 1 and 2 of the workgroup are inside; every wavefront calls it
    __device__ __forceinline__ void run(Lds& s, const SsaArgs<T>& a, const T* __restrict__ pdu,
                                        const T* __restrict__ pdv, const T* __restrict__ pdH, T calving_rate, int w,
                                        int lane, int i, int j) {
        const int ny = a.ny, nx = a.nx;
        const T D = a.dxi, hD = T(0.5) * D;
        const int jc = clampi(j, 0, nx - 1), ju = clampi(j, 0, nx);
        const int ic = clampi(i, 0, ny - 1);
        const long rc = (long)ic * nx, rf = (long)ic * (nx + 1);
        const long rft = (long)clampi(i - 1, 0, ny - 1) * (nx + 1), rfb = (long)clampi(i + 1, 0, ny - 1) * (nx + 1);
        const long rv0 = (long)clampi(i, 0, ny) * nx, rv1 = (long)clampi(i + 1, 0, ny) * nx;
        u = (a.u + rf)[ju];
        const T ut = (a.u + rft)[ju], ub = (a.u + rfb)[ju];
        v = (a.v + rv0)[jc];
        const T vb = (a.v + rv1)[jc];
        H = (a.H + rc)[jc];
        phi = (a.phi + rc)[jc];
        const T bed = (a.bed + rc)[jc], beta = (a.beta + rc)[jc], B = (a.B + rc)[jc];
        T du = T(0), dut = T(0), dub = T(0), dv = T(0), dvb = T(0);
        dH = T(0);
        if constexpr (JVP) {
            du = (pdu + rf)[ju];
            dut = (pdu + rft)[ju];
            dub = (pdu + rfb)[ju];
            dv = (pdv + rv0)[jc];
            dvb = (pdv + rv1)[jc];
            dH = (pdH + rc)[jc];
        }
        const bool jin = j > 0 && j < nx;
        const bool vt_in = jin && i > 0 && i < ny, vb_in = jin && i + 1 > 0 && i + 1 < ny;
        const T vl = lane_left(v), vbl = lane_left(vb), ur = lane_right(u);
        const T et = vt_in ? hD * ((ut - u) + (v - vl)) : T(0);
        const T eb = vb_in ? hD * ((u - ub) + (vb - vbl)) : T(0);
        const T exx = (ur - u) * D, eyy = (v - vb) * D;
        const T qs = et * et + eb * eb;
        const T sx = T(2) * exx + eyy, sy = exx + T(2) * eyy;
        const T e2 = exx * exx + eyy * eyy + exx * eyy + T(0.25) * (qs + lane_right(qs)) + a.P.eps_reg;
        const T eta = T(0.5) * B * glen_power(e2, a.P);
        const T eH = eta * H;
        const T g = T(1) - (T(1) - phi) * T(0.917);
        const T S = phi * bed + g * H, bp = beta * phi;
        // normal stresses (JVP: their derivatives) and the derivative of eta H
        T Sxx = T(2) * eH * sx, Syy = T(2) * eH * sy, dt_ = T(0), deH = T(0), dvl = T(0), dvbl = T(0), dur = T(0);
        if constexpr (JVP) {
            dvl = lane_left(dv);
            dvbl = lane_left(dvb);
            dur = lane_right(du);
            dt_ = vt_in ? hD * ((dut - du) + (dv - dvl)) : T(0);
            const T db = vb_in ? hD * ((du - dub) + (dvb - dvbl)) : T(0);
            const T dxx = (dur - du) * D, dyy = (dv - dvb) * D;
            const T ws = et * dt_ + eb * db;
            const T de2 = sx * dxx + sy * dyy + T(0.5) * (ws + lane_right(ws));
            deH = eH * (a.P.glen_p * de2) * row_rcp(e2) + eta * dH;
            Sxx = T(2) * (eH * (T(2) * dxx + dyy) + sx * deH);
            Syy = T(2) * (eH * (dxx + T(2) * dyy) + sy * deH);
        }
        {
            T(*p)[kRowLanes] = s.up[w];
            p[0][lane] = eH; p[1][lane] = Syy; p[2][lane] = H; p[3][lane] = S; p[4][lane] = bp;
            if constexpr (JVP) { p[kUp - 3][lane] = deH; p[kUp - 2][lane] = dH; p[kUp - 1][lane] = g; }
        }

        // u facet (i, j) but for the shear of its vertices, and its mass flux
        T Fx = T(0);
        {
            const T Hl = lane_left(H), Sl = lane_left(S), Sxl = lane_left(Sxx), be = T(0.5) * (lane_left(bp) + bp);
            const T sp = u * u + T(10), rs = row_rsqrt(sp), al = sp * rs, Hm = T(0.5) * (Hl + H);
            T pw = T(1), dpw = T(0);
            if (DRAG && w > 0 && w < NW - 1) {  // the halo rows need no drag
                const T z = u * u + T(0.25) * (vl * vl + v * v + vbl * vbl + vb * vb) + a.P.u_reg;
                pw = pow(z, a.P.drag_q);
                if constexpr (JVP) dpw = a.P.drag_q * pow(z, a.P.drag_q - T(1));
            }
            if constexpr (JVP) {
                const T dHl = lane_left(dH), gl = lane_left(g);
                if (jin) Fx = (Hm - T(0.5) * (u * rs) * (H - Hl)) * du + T(0.5) * ((u + al) * dHl + (u - al) * dH);
                ru = (Sxx - Sxl) * D - (be * (T(2) * dpw * u * u + pw) + a.P.water_drag) * du;
                if constexpr (DRAG) ru -= be * T(0.5) * dpw * u * (vl * dvl + v * dv + vbl * dvbl + vb * dvb);
                ru -= (T(0.5) * (dHl + dH) * (S - Sl) + Hm * (g * dH - gl * dHl)) * D;
            } else {
                if (jin) Fx = Hm * u - T(0.5) * al * (H - Hl);
                ru = (Sxx - Sxl) * D - (be * pw + a.P.water_drag) * u - Hm * (S - Sl) * D;
            }
        }
        __syncthreads();

        // the top-left vertex and the v facet (i, j)
        T Txy = T(0), Fy = T(0);
        rv = T(0);
        if (w > 0) {
            const T(*p)[kRowLanes] = s.up[w - 1];
            const T eHs = eH + p[0][lane], Syt = p[1][lane], Ht = p[2][lane], St = p[3][lane];
            const T be = T(0.5) * (p[4][lane] + bp);
            const T eHv = T(0.25) * (eHs + lane_left(eHs));
            T deHs = T(0), dHt = T(0), gt = T(0);
            if constexpr (JVP) { deHs = deH + p[kUp - 3][lane]; dHt = p[kUp - 2][lane]; gt = p[kUp - 1][lane]; }
            if constexpr (JVP) Txy = T(2) * (eHv * dt_ + et * (T(0.25) * (deHs + lane_left(deHs))));
            else Txy = T(2) * eHv * et;
            const T Txr = lane_right(Txy);  // zero beyond the domain's vertices
            const T sp = v * v + T(10), rs = row_rsqrt(sp), al = sp * rs, Hm = T(0.5) * (Ht + H);
            const bool iin = i > 0 && i < ny;
            T pw = T(1), dpw = T(0);
            if (DRAG && w < NW - 1) {
                const T utr = lane_right(ut);
                const T z = v * v + T(0.25) * (ut * ut + utr * utr + u * u + ur * ur) + a.P.u_reg;
                pw = pow(z, a.P.drag_q);
                if constexpr (JVP) dpw = a.P.drag_q * pow(z, a.P.drag_q - T(1));
            }
            if constexpr (JVP) {
                if (iin) Fy = (Hm - T(0.5) * (v * rs) * (Ht - H)) * dv + T(0.5) * ((v - al) * dHt + (v + al) * dH);
                rv = (Syt - Syy) * D + (Txr - Txy) * D - (be * (T(2) * dpw * v * v + pw) + a.P.water_drag) * dv;
                if constexpr (DRAG) {
                    const T utr = lane_right(ut), dutr = lane_right(dut);
                    rv -= be * T(0.5) * dpw * v * (ut * dut + utr * dutr + u * du + ur * dur);
                }
                rv -= (T(0.5) * (dHt + dH) * (St - S) + Hm * (gt * dHt - g * dH)) * D;
            } else {
                if (iin) Fy = Hm * v - T(0.5) * al * (Ht - H);
                rv = (Syt - Syy) * D + (Txr - Txy) * D - (be * pw + a.P.water_drag) * v - Hm * (St - S) * D;
            }
            s.down[w][0][lane] = Txy;
            s.down[w][1][lane] = Fy;
        }
        __syncthreads();

        rH = T(0);
        if (w > 0 && w < NW - 1) {
            const T(*q)[kRowLanes] = s.down[w + 1];
            ru += (Txy - q[0][lane]) * D;
            const T Hq = JVP ? dH : H;
            rH = Hq / a.dt + ((lane_right(Fx) - Fx) + (Fy - q[1][lane])) * D;
            if (calving_rate != T(0)) {
                const long rt = (long)clampi(ic - 1, 0, ny - 1) * nx, rb = (long)clampi(ic + 1, 0, ny - 1) * nx;
                const int jl = clampi(jc - 1, 0, nx - 1), jr = clampi(jc + 1, 0, nx - 1);
                const T k = (T(1) - phi) * ((T(1) - (a.phi + rc)[jl]) + (T(1) - (a.phi + rc)[jr]) +
                                            (T(1) - (a.phi + rt)[jc]) + (T(1) - (a.phi + rb)[jc]));
                rH += k * calving_rate * Hq * D;
            }
        }
    }
};

}  // namespace glide
