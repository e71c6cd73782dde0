// gfx950 kernels of the multicolour (red-black) Vanka smoother, the smoother
// of the mixed-precision solver (no counterpart in the reference, whose Vanka
// pass is additive: glide/cuda/vanka.cu:477-660).
//
// A pass takes the cell viscosity of the state it starts from (frozen for the
// pass, as in the reference), solves the red cells ((i + j) even) and then the
// black ones; each facet belongs to exactly one cell of a colour.  Cells of one
// colour read each other's old values, so a colour is a block-Jacobi step over
// non-overlapping patches and the result does not depend on scheduling
// (run-to-run bitwise identical).
//
// k_mc_pass: the whole pass in one launch, from one buffer set into another.
// A workgroup updates 58 columns and 2 NW - 2 rows (NW wavefronts).  It loads
// the state three cells around them into LDS, one wavefront per row, and forms
// the viscosity; then a half wavefront owns a row and a lane a cell pair: it
// solves the red cells of the tile and of a ring of one cell around it (what a
// black cell reads of another cell was written by the red cells beside it, or
// is old), puts them back into LDS, and solves the black cells.  The local
// Newton iteration runs the folded cell system of the additive smoother
// (cell_system, refined hardware reciprocals), without compensated updates and
// with the caller's relaxation and stopping threshold.
//
// k_cell_eta, k_mc_phase: the same pass as a launch for the viscosity and one per
// colour, for heavy local solves on large levels (mc_phases_faster).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "row_ops.hpp"
#include "ssa_device.hpp"
#include "ssa_kernels.hpp"
#include "tab.hpp"

namespace glide {

namespace {

constexpr int kMcCols = kRowLanes - 6;  // columns a workgroup updates

// rows rr = 0 .. kF - 1 of u and v are the tile's rows -3 .. kRows + 2, rows
// 0 .. kC - 1 of the cell planes its rows -2 .. kRows + 1; column l is the
// tile's column l - 3.
template <typename T, int NW>
struct McLds {
    static constexpr int kRows = 2 * NW - 2, kF = kRows + 6, kC = kRows + 4;
    T u[kF][kRowLanes], v[kF][kRowLanes];
    T H[kC][kRowLanes], eH[kC][kRowLanes], eta[kC][kRowLanes];
    T S[kC][kRowLanes], bp[kC][kRowLanes], phi[kC][kRowLanes];  // flotation surface, beta * phi
};

// What a cell's solve reads of its own cell only.
template <typename T>
struct McCentre {
    T f[5], bed, thk;
    __device__ __forceinline__ void load(const SsaArgs<T>& a, int i, int j) {
        const long c = (long)i * a.nx + j, ou = c + i;
        if (a.f_u) {
            f[0] = a.f_u[ou]; f[1] = a.f_u[ou + 1];
            f[2] = a.f_v[c]; f[3] = a.f_v[c + a.nx];
            f[4] = a.f_H[c];
        } else {
            f[0] = f[1] = f[2] = f[3] = f[4] = T(0);
        }
        bed = a.bed[c];
        thk = a.gamma ? a.gamma[c] : T(0);
    }
};

// The folded system of the cell at LDS row rr, column c (grid cell (i, j)) for
// the state in LDS; its viscosity comes back in e_c.  EDGE: the cell may lie on
// the domain edge.
template <typename T, bool LINEAR, bool EDGE, class L>
__device__ __forceinline__ void mc_cell_sys(CellSys<T>& cs, const L& s, const SsaArgs<T>& a, const McCentre<T>& q,
                                            const VankaArgs<T>& vk, int rr, int c, int i, int j, T& e_c) {
    const int ny = a.ny, nx = a.nx, k = rr - 1;
    const bool il = !EDGE || j > 0, ir = !EDGE || j + 1 < nx, it_ = !EDGE || i > 0, ib = !EDGE || i + 1 < ny;
    const T D = a.dxi, D2 = D * D;
    const T e_l = s.eH[k][c - 1], e_r = s.eH[k][c + 1], e_t = s.eH[k - 1][c], e_b = s.eH[k + 1][c];
    e_c = s.eta[k][c];
    cs.D = D;
    cs.hD = T(0.5) * D;
    cs.H_l = s.H[k][c - 1]; cs.H_r = s.H[k][c + 1]; cs.H_t = s.H[k - 1][c]; cs.H_b = s.H[k + 1][c];
    cs.dL = il ? D : T(0); cs.dR = ir ? D : T(0); cs.dT = it_ ? D : T(0); cs.dB = ib ? D : T(0);
    const T p_c = s.phi[k][c];
    T kcal = T(0);
    if (vk.calving_rate != T(0))
        kcal = (T(1) - p_c) * vk.calving_rate *
               ((T(1) - s.phi[k][c - 1]) + (T(1) - s.phi[k][c + 1]) + (T(1) - s.phi[k - 1][c]) +
                (T(1) - s.phi[k + 1][c]));
    cs.r4h = T(1) / a.dt + kcal * D;
    cs.j24c = cs.r4h + vk.mc_damping;
    cs.f4 = q.f[4];
    cs.kH = T(2) * e_c * D2;
    const T qc = T(0.25) * e_c;
    const bool vtl = it_ && il, vtr = it_ && ir, vbl = ib && il, vbr = ib && ir;
    cs.C_tl = vtl ? T(0.25) * (s.eH[k - 1][c - 1] + e_t + e_l) : T(0);
    cs.C_tr = vtr ? T(0.25) * (e_t + s.eH[k - 1][c + 1] + e_r) : T(0);
    cs.C_bl = vbl ? T(0.25) * (e_l + s.eH[k + 1][c - 1] + e_b) : T(0);
    cs.C_br = vbr ? T(0.25) * (e_r + e_b + s.eH[k + 1][c + 1]) : T(0);
    cs.q_tl = vtl ? qc : T(0); cs.q_tr = vtr ? qc : T(0); cs.q_bl = vbl ? qc : T(0); cs.q_br = vbr ? qc : T(0);
    cs.u_tl = s.u[rr - 1][c]; cs.u_tr = s.u[rr - 1][c + 1];
    cs.u_bl = s.u[rr + 1][c]; cs.u_br = s.u[rr + 1][c + 1];
    cs.v_lt = s.v[rr][c - 1]; cs.v_lb = s.v[rr + 1][c - 1];
    cs.v_rt = s.v[rr][c + 1]; cs.v_rb = s.v[rr + 1][c + 1];
    cs.s_tl = cs.hD * (cs.u_tl - cs.v_lt);
    cs.s_tr = cs.hD * (cs.u_tr + cs.v_rt);
    cs.s_bl = -cs.hD * (cs.u_bl + cs.v_lb);
    cs.s_br = cs.hD * (cs.v_rb - cs.u_br);
    const T nl = il ? T(2) * e_l * D2 : T(0), nr = ir ? T(2) * e_r * D2 : T(0);
    const T nt = it_ ? T(2) * e_t * D2 : T(0), nb = ib ? T(2) * e_b * D2 : T(0);
    cs.c0 = -nl * (cs.v_lt - cs.v_lb - T(2) * s.u[rr][c - 1]) - q.f[0];
    cs.c1 = nr * (T(2) * s.u[rr][c + 2] + cs.v_rt - cs.v_rb) - q.f[1];
    cs.c2 = nt * (cs.u_tr - cs.u_tl + T(2) * s.v[rr - 1][c]) - q.f[2];
    cs.c3 = -nb * (cs.u_br - cs.u_bl - T(2) * s.v[rr + 2][c]) - q.f[3];
    const T b_c = s.bp[k][c];
    cs.be_l = T(0.5) * (s.bp[k][c - 1] + b_c);
    cs.be_r = T(0.5) * (b_c + s.bp[k][c + 1]);
    cs.be_t = T(0.5) * (s.bp[k - 1][c] + b_c);
    cs.be_b = T(0.5) * (b_c + s.bp[k + 1][c]);
    const T lin = LINEAR ? T(1) : T(0), wd = a.P.water_drag;
    cs.o0 = -T(2) * nl - lin * (cs.be_l + wd);
    cs.o1 = -T(2) * nr - lin * (cs.be_r + wd);
    cs.o2 = -T(2) * nt - lin * (cs.be_t + wd);
    cs.o3 = -T(2) * nb - lin * (cs.be_b + wd);
    cs.a0 = cs.o0 - (cs.C_tl + cs.C_bl) * D2 - vk.ssa_damping;
    cs.a1 = cs.o1 - (cs.C_tr + cs.C_br) * D2 - vk.ssa_damping;
    cs.a2 = cs.o2 - (cs.C_tl + cs.C_tr) * D2 - vk.ssa_damping;
    cs.a3 = cs.o3 - (cs.C_bl + cs.C_br) * D2 - vk.ssa_damping;
    cs.h0 = -(cs.q_tl + cs.q_bl) * D2;
    cs.h1 = -(cs.q_tr + cs.q_br) * D2;
    cs.h2 = -(cs.q_tl + cs.q_tr) * D2;
    cs.h3 = -(cs.q_bl + cs.q_br) * D2;
    cs.eD = T(2) * e_c * D;
    cs.S_l = s.S[k][c - 1]; cs.S_r = s.S[k][c + 1]; cs.S_t = s.S[k - 1][c]; cs.S_b = s.S[k + 1][c];
    cs.Zc = p_c * q.bed;
    cs.gc = T(1) - (T(1) - p_c) * T(0.917);
}

// Local Newton iteration of the cell at LDS row rr, column c (grid cell (i, j))
// against the state in LDS: the new unknowns x, the active-set flag, and the
// cell's viscosity and surface coefficients.  EDGE: the cell may lie on the
// domain edge (the Dirichlet pins are tested).
template <typename T, int NW, bool LINEAR, bool EDGE>
__device__ __forceinline__ void mc_newton(const McLds<T, NW>& s, const SsaArgs<T>& a, const McCentre<T>& q,
                                          const VankaArgs<T>& vk, bool solves, int rr, int c, int i, int j, T x[5],
                                          T& masked, T& e_c, T& Zc, T& gc) {
    const int ny = a.ny, nx = a.nx, k = rr - 1;
    CellSys<T> cs;
    mc_cell_sys<T, LINEAR, EDGE>(cs, s, a, q, vk, rr, c, i, j, e_c);
    Zc = cs.Zc;
    gc = cs.gc;
    const T thk = q.thk;
    x[0] = s.u[rr][c];
    x[1] = s.u[rr][c + 1];
    x[2] = s.v[rr][c];
    x[3] = s.v[rr + 1][c];
    x[4] = s.H[k][c];
    const bool pin0 = EDGE && j == 0, pin1 = EDGE && j == nx - 1, pin2 = EDGE && i == 0, pin3 = EDGE && i == ny - 1;
    // every lane iterates as long as one of the wavefront does: a wavefront with
    // few lanes left in its execution mask issues the same instructions at a
    // third of the rate (12 steps at 12 x 59 cells: 61 us against 24 us)
    bool go = solves && vk.newton_steps > 0 && T(1e30) > vk.tol;
    for (int it = 1; __any(go); ++it) {
        T J[25], r[5];
        cell_system<T, T, LINEAR>(cs, cs, x, J, r, a.P);
        if constexpr (EDGE) {
            if (pin0) { pin_row(J, 0); r[0] = x[0]; }
            if (pin1) { pin_row(J, 1); r[1] = x[1]; }
            if (pin2) { pin_row(J, 2); r[2] = x[2]; }
            if (pin3) { pin_row(J, 3); r[3] = x[3]; }
        }
        const bool pin4 = (x[4] - a.dt * r[4]) <= thk;
        if (pin4) {
            pin_row(J, 4);
            r[4] = x[4] - thk;
        }
        T d[5];
        lu5_solve_rcp(J, r, d);
        const T rnorm = r[0] * r[0] + r[1] * r[1] + r[2] * r[2] + r[3] * r[3] + r[4] * r[4];
#pragma unroll
        for (int k2 = 0; k2 < 5; ++k2) {
            const T y = x[k2] - vk.relax * d[k2];
            x[k2] = go ? (k2 == 4 ? fmax(y, thk) : y) : x[k2];
        }
        masked = go ? (pin4 ? T(1) : T(0)) : masked;
        go = go && it < vk.newton_steps && rnorm > vk.tol;
    }
}

template <typename T, int NW, bool LINEAR>
__device__ __forceinline__ void mc_pass_body(int bx, int by, const SsaArgs<T>& a, T* __restrict__ u_dst,
                                             T* __restrict__ v_dst, T* __restrict__ H_dst, T* __restrict__ mask,
                                             T* __restrict__ phi_dst, const VankaArgs<T>& vk) {
    using L = McLds<T, NW>;
    __shared__ L s;
    const int ny = a.ny, nx = a.nx;
    const int lane = threadIdx.x, w = wave_row(threadIdx.y);
    const int i0 = by * L::kRows, j0 = bx * kMcCols;

    // this thread's cell of a colour: its tile row r (red: also the rows -1 and
    // kRows of the ring) and column c; the last wavefront has no black row
    auto place = [&](int colour, int& r, int& c) -> bool {
        r = 2 * w + (lane >> 5) - 1 + colour;
        const int i = i0 + r, lo = colour ? 0 : -1, hi = kMcCols - lo;
        c = lo + 2 * (lane & 31) + ((i + lo + colour) & 1);  // j0 is even
        return i >= 0 && i < ny && r < L::kRows - lo && c < hi && j0 + c >= 0 && j0 + c < nx;
    };
    int r, c;
    bool solves = place(0, r, c);
    McCentre<T> q{};
    if (solves) q.load(a, i0 + r, j0 + c);

    // the tile's rows, one wavefront each: state, surface, drag, viscosity; all
    // loads are issued before the first is used
    constexpr int kIt = (L::kF + NW - 1) / NW;
    T u_[kIt], v_[kIt], H_[kIt], B_[kIt], z_[kIt], b_[kIt], p_[kIt];
    const int j = j0 - 3 + lane, jc = clampi(j, 0, nx - 1), ju = clampi(j, 0, nx);
#pragma unroll
    for (int t = 0; t < kIt; ++t) {
        const int ir = i0 - 3 + w + t * NW, ic = clampi(ir, 0, ny - 1);
        const long rc = (long)ic * nx;
        u_[t] = (a.u + rc + ic)[ju];
        v_[t] = (a.v + (long)clampi(ir, 0, ny) * nx)[jc];
        H_[t] = (a.H + rc)[jc];
        B_[t] = (a.B + rc)[jc];
        z_[t] = (a.bed + rc)[jc];
        b_[t] = (a.beta + rc)[jc];
        p_[t] = phi_dst ? T(0) : (a.phi + rc)[jc];
    }
#pragma unroll
    for (int t = 0; t < kIt; ++t) {
        const int rr = w + t * NW;
        if (rr < L::kF) {
            s.u[rr][lane] = u_[t];
            s.v[rr][lane] = v_[t];
        }
        if (rr >= 1 && rr <= L::kC) {
            const int ir = i0 - 3 + rr;
            const T H = H_[t];
            T p = p_[t];
            if (phi_dst) {
                p = grounded_fraction(H, z_[t], a.P.frd);
                if (ir >= 0 && ir < ny && rr >= 3 && rr < 3 + L::kRows && lane >= 3 && lane < 3 + kMcCols && j < nx)
                    (phi_dst + (long)ir * nx)[j] = p;
            }
            s.H[rr - 1][lane] = H;
            s.phi[rr - 1][lane] = p;
            s.S[rr - 1][lane] = p * z_[t] - (T(1) - p) * T(0.917) * H + H;
            s.bp[rr - 1][lane] = b_[t] * p;
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kIt; ++t) {
        const int rr = w + t * NW;
        if (rr >= 1 && rr <= L::kC) {
            const int ir = i0 - 3 + rr;
            const bool jin = j > 0 && j < nx;
            const bool vt_in = jin && ir > 0 && ir < ny, vb_in = jin && ir + 1 > 0 && ir + 1 < ny;
            const T u = u_[t], v = v_[t], vb = s.v[rr + 1][lane];
            const T hD = T(0.5) * a.dxi;
            const T vl = lane_left(v), vbl = lane_left(vb);
            const T et = vt_in ? hD * ((s.u[rr - 1][lane] - u) + (v - vl)) : T(0);
            const T eb = vb_in ? hD * ((u - s.u[rr + 1][lane]) + (vb - vbl)) : T(0);
            const T qs = et * et + eb * eb;
            const T exx = (lane_right(u) - u) * a.dxi, eyy = (v - vb) * a.dxi;
            const T e2 = exx * exx + eyy * eyy + exx * eyy + T(0.25) * (qs + lane_right(qs)) + a.P.eps_reg;
            const T eta = T(0.5) * B_[t] * glen_power(e2, a.P);
            s.eta[rr - 1][lane] = eta;
            s.eH[rr - 1][lane] = eta * H_[t];
        }
    }
    __syncthreads();

    const bool stepped = vk.newton_steps > 0 && T(1e30) > vk.tol;
#pragma unroll 1
    for (int colour = 0; colour < 2; ++colour) {
        // the black cell's own values are loaded ahead of the red solve
        int rn = 0, cn = 0;
        const bool next = colour == 0 && place(1, rn, cn);
        McCentre<T> qn{};
        if (next) qn.load(a, i0 + rn, j0 + cn);
        // wavefronts whose rows or columns touch the domain edge test the pins
        const int it = i0 + 2 * w - 1 + colour;
        const bool edge = it <= 0 || it + 1 >= ny - 1 || bx == 0 || j0 + kMcCols >= nx - 1;
        // lanes without a cell compute along inside the tile
        const int i = i0 + r, j = j0 + c, rr = min(r, L::kRows) + 3, l = min(c, kMcCols) + 3;
        T x[5], masked = T(0), e_c = T(0), Zc = T(0), gc = T(0);
        if (__any(solves)) {
            if (edge) mc_newton<T, NW, LINEAR, true>(s, a, q, vk, solves, rr, l, i, j, x, masked, e_c, Zc, gc);
            else mc_newton<T, NW, LINEAR, false>(s, a, q, vk, solves, rr, l, i, j, x, masked, e_c, Zc, gc);
        }
        const long o = (long)i * nx + j, ou = o + i;
        const bool own = solves && r >= 0 && r < L::kRows && c >= 0 && c < kMcCols;
        if (own) {
            H_dst[o] = x[4];
            if (stepped) mask[o] = masked;
            // black cells write the facets; the domain's edge facets of a red
            // cell have no black cell
            if (colour == 1 || j == 0) u_dst[ou] = x[0];
            if (colour == 1 || j == nx - 1) u_dst[ou + 1] = x[1];
            if (colour == 1 || i == 0) v_dst[o] = x[2];
            if (colour == 1 || i == ny - 1) v_dst[o + nx] = x[3];
        }
        if (colour == 1) break;
        __syncthreads();
        if (solves) {
            s.u[rr][l] = x[0];
            s.u[rr][l + 1] = x[1];
            s.v[rr][l] = x[2];
            s.v[rr + 1][l] = x[3];
            s.H[rr - 1][l] = x[4];
            s.eH[rr - 1][l] = e_c * x[4];
            s.S[rr - 1][l] = Zc + gc * x[4];
        }
        __syncthreads();
        r = rn; c = cn;
        solves = next;
        q = qn;
    }
}

template <typename T, int NW, bool LINEAR>
__global__ __launch_bounds__(kRowLanes* NW) void k_mc_pass(SsaArgs<T> a, T* __restrict__ u_dst,
                                                           T* __restrict__ v_dst, T* __restrict__ H_dst,
                                                           T* __restrict__ mask, T* __restrict__ phi_dst,
                                                           VankaArgs<T> vk, int gx) {
    const int b = xcd_block(blockIdx.x, gridDim.x);
    mc_pass_body<T, NW, LINEAR>(b % gx, b / gx, a, u_dst, v_dst, H_dst, mask, phi_dst, vk);
}

// The pass in three launches, for levels that fill the device with heavy local
// solves (mc_phases_faster): the viscosity, then a launch per colour, from one
// buffer set into the other.  A lane owns a cell of the colour and the other cell
// beside it, so a wavefront covers 128 columns and no cell is solved twice: the
// one-launch form solves 8 rows of red cells for every 6 and leaves 3 lanes of 32
// and a wavefront of 4 idle in turn.
template <typename T>
__global__ __launch_bounds__(256) void k_cell_eta(SsaArgs<T> a, T* __restrict__ eta) {
    const int j = blockIdx.x * 256 + threadIdx.x, i = blockIdx.y;
    if (j >= a.nx) return;
    const CellVel<T> c = load_cell_vel<T>(a.u, a.v, i, j, a.ny, a.nx);
    const T e2 = strain_invariant(c, i, j, a.ny, a.nx, a.dxi, a.P.eps_reg);
    eta[(long)i * a.nx + j] = T(0.5) * a.B[(long)i * a.nx + j] * glen_power(e2, a.P);
}

// Local Newton iteration of cell (i, j) against the state in a; returns the
// new unknowns x and the active-set flag.  EDGE: the cell may lie on the
// domain edge (the Dirichlet pins are tested).
template <typename T, bool LINEAR, bool EDGE>
__device__ __forceinline__ void phase_newton(const SsaArgs<T>& a, const T* __restrict__ eta, int i, int j,
                                             const VankaArgs<T>& vk, T x[5], T& masked) {
    const int ny = a.ny, nx = a.nx;
    CellSys<T> cs;
    T thk;
    {
        Patch<T> p;
        load_patch_with<T>(p, a, [&](int di, int dj) { return eta[offC(i + di, j + dj, ny, nx)]; }, i, j, a.f_u, a.f_v,
                           a.f_H, a.phi);
        make_cell_sys(cs, p, a.P, vk.calving_rate, a.dxi, a.dt, vk.ssa_damping, vk.mc_damping);
        thk = p.gam;
    }
    const long c = (long)i * nx + j;
    x[0] = a.u[(long)i * (nx + 1) + j];
    x[1] = a.u[(long)i * (nx + 1) + j + 1];
    x[2] = a.v[c];
    x[3] = a.v[c + nx];
    x[4] = a.H[c];
    const bool pin0 = j == 0, pin1 = j == nx - 1, pin2 = i == 0, pin3 = i == ny - 1;
    T rnorm = T(1e30);
    for (int it = 0; it < vk.newton_steps && rnorm > vk.tol; ++it) {
        T J[25], r[5];
        cell_system<T, T, LINEAR>(cs, cs, x, J, r, a.P);
        if constexpr (EDGE) {
            if (pin0) { pin_row(J, 0); r[0] = x[0]; }
            if (pin1) { pin_row(J, 1); r[1] = x[1]; }
            if (pin2) { pin_row(J, 2); r[2] = x[2]; }
            if (pin3) { pin_row(J, 3); r[3] = x[3]; }
        }
        if ((x[4] - a.dt * r[4]) <= thk) {
            masked = T(1);
            pin_row(J, 4);
            r[4] = x[4] - thk;
        } else {
            masked = T(0);
        }
        T d[5];
        lu5_solve_rcp(J, r, d);
        rnorm = r[0] * r[0] + r[1] * r[1] + r[2] * r[2] + r[3] * r[3] + r[4] * r[4];
#pragma unroll
        for (int k = 0; k < 5; ++k) x[k] -= vk.relax * d[k];
        x[4] = fmax(x[4], thk);
    }
}

constexpr int kPhaseRows = 4;  // rows per block
template <typename T, bool LINEAR>
__global__ __launch_bounds__(kRowLanes* kPhaseRows) void k_mc_phase(SsaArgs<T> a, const T* __restrict__ eta,
                                                                    T* __restrict__ u_dst, T* __restrict__ v_dst,
                                                                    T* __restrict__ H_dst, T* __restrict__ mask,
                                                                    VankaArgs<T> vk, int colour) {
    const int ny = a.ny, nx = a.nx;
    const int bx = blockIdx.x, i = blockIdx.y * kPhaseRows + threadIdx.y;
    if (i >= ny) return;
    const int pair = bx * kRowLanes + threadIdx.x;
    const int p = (i + colour) & 1;
    const int j = 2 * pair + p;       // the lane's cell of the colour
    const int jo = 2 * pair + 1 - p;  // and the other one beside it
    if (j < nx) {
        const long c = (long)i * nx + j;
        T x[5], masked = mask[c];
        const bool edge = i == 0 || i == ny - 1 || bx == 0 || 2 * (bx + 1) * kRowLanes >= nx;
        if (edge) phase_newton<T, LINEAR, true>(a, eta, i, j, vk, x, masked);
        else phase_newton<T, LINEAR, false>(a, eta, i, j, vk, x, masked);
        u_dst[(long)i * (nx + 1) + j] = x[0];
        u_dst[(long)i * (nx + 1) + j + 1] = x[1];
        v_dst[c] = x[2];
        v_dst[c + nx] = x[3];
        H_dst[c] = x[4];
        mask[c] = masked;
    }
    if (jo < nx) {
        const long c = (long)i * nx + jo;
        H_dst[c] = a.H[c];
        if (jo == 0) u_dst[(long)i * (nx + 1)] = a.u[(long)i * (nx + 1)];
        if (jo == nx - 1) u_dst[(long)i * (nx + 1) + nx] = a.u[(long)i * (nx + 1) + nx];
        if (i == 0) v_dst[jo] = a.v[jo];
        if (i == ny - 1) v_dst[(long)ny * nx + jo] = a.v[(long)ny * nx + jo];
    }
}

// All additive forward passes of a level of at most 16 x 16 cells in one
// workgroup, the state in LDS: 16 lanes a row, four rows a wavefront, one
// wavefront per SIMD.  A pass of k_vanka_persistent reads the level's state and
// parameters through the L2 twice (viscosity, then patches) and meets other
// workgroups at a barrier; most passes of the coarsest level run one or two
// Newton iterations, so that this was most of a pass (14 x 14: 5.9 us, here 3.5).
constexpr int kTinySide = 16;
template <typename T>
struct TinyLds {  // the planes of McLds for one tile of 16 x 16
    static constexpr int kF = kTinySide + 6, kC = kTinySide + 4;
    T u[kF][kF], v[kF][kF];
    T H[kC][kF], eH[kC][kF], eta[kC][kF], S[kC][kF], bp[kC][kF], phi[kC][kF];
    T w3[kTinySide + 1][kTinySide];  // bottom-facet increments of row r at r + 1
};
template <bool LINEAR>
__global__ __launch_bounds__(kTinySide* kTinySide, 1) void k_vanka_tiny(SsaArgs<double> a, double* __restrict__ pu,
                                                                        double* __restrict__ pv,
                                                                        double* __restrict__ pH,
                                                                        double* __restrict__ mask,
                                                                        VankaArgs<double> vk, double omega,
                                                                        int n_iter) {
    using T = double;
    using L = TinyLds<T>;
    __shared__ L s;
    const int ny = a.ny, nx = a.nx, tid = threadIdx.x;
    const int j = tid & (kTinySide - 1), i = tid >> 4, rr = i + 3, c = j + 3, k = rr - 1;
    const bool cell = i < ny && j < nx;
    for (int q = tid; q < L::kF * L::kF; q += kTinySide * kTinySide) {
        const int r = q / L::kF, l = q % L::kF;
        const int ri = clampi(r - 3, 0, ny - 1), lj = clampi(l - 3, 0, nx - 1);
        s.u[r][l] = pu[ri * (nx + 1) + clampi(l - 3, 0, nx)];
        s.v[r][l] = pv[clampi(r - 3, 0, ny) * nx + lj];
        if (r >= 1 && r <= L::kC) {
            const int o = ri * nx + lj;
            const T H = pH[o], p = a.phi[o];
            s.H[r - 1][l] = H;
            s.phi[r - 1][l] = p;
            s.S[r - 1][l] = p * a.bed[o] - (T(1) - p) * T(0.917) * H + H;
            s.bp[r - 1][l] = a.beta[o] * p;
            s.eH[r - 1][l] = T(0);
            s.eta[r - 1][l] = T(0);
        }
    }
    if (tid < kTinySide) s.w3[0][tid] = T(0);
    const int ic = min(i, ny - 1), jc = min(j, nx - 1);
    McCentre<T> q{};
    q.load(a, ic, jc);
    const T B = a.B[ic * nx + jc];
    T masked = mask[ic * nx + jc];
    const bool jin = j > 0 && j < nx, vt_in = jin && i > 0 && i < ny, vb_in = jin && i + 1 < ny;
    const bool pin0 = j == 0, pin1 = j == nx - 1, pin2 = i == 0, pin3 = i == ny - 1;
    const T D = a.dxi, hD = T(0.5) * D, tol = T(1e-6);
    __syncthreads();
#pragma unroll 1
    for (int pass = 0; pass < n_iter; ++pass) {
        {
            const T u = s.u[rr][c], v = s.v[rr][c], vb = s.v[rr + 1][c];
            const T et = vt_in ? hD * ((s.u[rr - 1][c] - u) + (v - s.v[rr][c - 1])) : T(0);
            const T eb = vb_in ? hD * ((u - s.u[rr + 1][c]) + (vb - s.v[rr + 1][c - 1])) : T(0);
            const T qs = et * et + eb * eb, exx = (s.u[rr][c + 1] - u) * D, eyy = (v - vb) * D;
            const T e2 = exx * exx + eyy * eyy + exx * eyy + T(0.25) * (qs + lane16_right(qs)) + a.P.eps_reg;
            const T eta = T(0.5) * B * glen_power(e2, a.P);
            if (cell) {
                s.eta[k][c] = eta;
                s.eH[k][c] = eta * s.H[k][c];
            }
        }
        __syncthreads();
        const T x0[5] = {s.u[rr][c], s.u[rr][c + 1], s.v[rr][c], s.v[rr + 1][c], s.H[k][c]};
        T x[5] = {x0[0], x0[1], x0[2], x0[3], x0[4]}, cmp[5] = {T(0), T(0), T(0), T(0), T(0)};
        CellSys<T> cs;
        T e_c;
        mc_cell_sys<T, LINEAR, true>(cs, s, a, q, vk, rr, c, i, j, e_c);
        bool go = cell && vk.newton_steps > 0;
        int it = 0;
        while (__any(go)) {  // as cell_newton
            T J[25], r[5], d[5];
            cell_system<T, T, LINEAR>(cs, cs, x, J, r, a.P);
            if (pin0) { pin_row(J, 0); r[0] = x[0]; }
            if (pin1) { pin_row(J, 1); r[1] = x[1]; }
            if (pin2) { pin_row(J, 2); r[2] = x[2]; }
            if (pin3) { pin_row(J, 3); r[3] = x[3]; }
            const bool pin4 = (x[4] - a.dt * r[4]) <= q.thk;
            if (pin4) {
                pin_row(J, 4);
                r[4] = x[4] - q.thk;
            }
            masked = go ? (pin4 ? T(1) : T(0)) : masked;
            lu5_solve_rcp(J, r, d);
            const T rnorm = r[0] * r[0] + r[1] * r[1] + r[2] * r[2] + r[3] * r[3] + r[4] * r[4];
#pragma unroll
            for (int m = 0; m < 5; ++m) {  // compensated relaxed update, local relaxation 0.5
                const T y = T(-0.5) * d[m] - cmp[m];
                T t = x[m] + y;
                const T e = (t - x[m]) - y;
                if (m == 4) t = fmax(t, q.thk);
                cmp[m] = go ? e : cmp[m];
                x[m] = go ? t : x[m];
            }
            it += go ? 1 : 0;
            go = go && it < vk.newton_steps && rnorm > tol;
        }
        const T w0 = T(0.5) * (x[0] - x0[0]), w1 = cell ? T(0.5) * (x[1] - x0[1]) : T(0);
        const T w2 = T(0.5) * (x[2] - x0[2]), w3 = cell ? T(0.5) * (x[3] - x0[3]) : T(0);
        s.w3[i + 1][j] = w3;
        const T w1l = lane16_left(w1);
        __syncthreads();
        if (cell) {
            s.u[rr][c] = x0[0] + omega * (w0 + w1l);
            if (pin1) s.u[rr][c + 1] = x0[1] + omega * w1;
            s.v[rr][c] = x0[2] + omega * (w2 + s.w3[i][j]);
            if (pin3) s.v[rr + 1][c] = x0[3] + omega * w3;
            const T H = x0[4] + omega * (x[4] - x0[4]);
            s.H[k][c] = H;
            s.S[k][c] = cs.Zc + cs.gc * H;
        }
        __syncthreads();
    }
    if (cell) {
        const int o = i * nx + j;
        pu[o + i] = s.u[rr][c];
        if (pin1) pu[o + i + 1] = s.u[rr][c + 1];
        pv[o] = s.v[rr][c];
        if (pin3) pv[o + nx] = s.v[rr + 1][c];
        pH[o] = s.H[k][c];
        mask[o] = masked;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_pin_rows(T* __restrict__ du, T* __restrict__ dv, T* __restrict__ dH,
                                                  const T* __restrict__ mask, int ny, int nx) {
    const int i = blockIdx.y, j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j > nx) return;
    if (i < ny && (j == 0 || j == nx)) du[(long)i * (nx + 1) + j] = T(0);
    if (j < nx) {
        if (i == 0 || i == ny) dv[(long)i * nx + j] = T(0);
        if (i < ny && mask[(long)i * nx + j] > T(0.5)) dH[(long)i * nx + j] = T(0);
    }
}

}  // namespace

// The coarsest level's calls (200 passes), whose passes mostly take one or two
// Newton iterations: per pass at 14 x 14 in 200 passes 3.5 against 5.9 us.  The ten
// or twenty passes of another level are bound by their thirty iterations a cell,
// the same in both forms.  With four rows or fewer one wavefront holds the level.
bool vanka_tiny_fits(int ny, int nx, int n_iter) {
    return n_iter >= 32 && ny > 4 && ny <= kTinySide && nx >= 2 && nx <= kTinySide;
}
hipError_t launch_vanka_tiny(const SsaArgs<double>& a, double* u, double* v, double* H, double* mask,
                             const VankaArgs<double>& vk, double omega, int n_iter, hipStream_t st) {
    if (!vanka_tiny_fits(a.ny, a.nx, n_iter) || vk.local_fp32) return hipErrorInvalidValue;
    TimedLaunch tl(kTimeVankaCell, (long)a.ny * a.nx * n_iter, st);
    if (a.P.linear_drag)
        k_vanka_tiny<true><<<1, kTinySide * kTinySide, 0, st>>>(a, u, v, H, mask, vk, omega, n_iter);
    else
        k_vanka_tiny<false><<<1, kTinySide * kTinySide, 0, st>>>(a, u, v, H, mask, vk, omega, n_iter);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_pin_rows(T* du, T* dv, T* dH, const T* mask, int ny, int nx, hipStream_t st) {
    k_pin_rows<T><<<dim3((nx + 1 + 255) / 256, ny + 1), 256, 0, st>>>(du, dv, dH, mask, ny, nx);
    return hipGetLastError();
}

namespace {
int mc_blocks(int ny, int nx, int waves, int* gx) {
    const int rows = 2 * waves - 2;
    *gx = (nx + kMcCols - 1) / kMcCols;
    return *gx * ((ny + rows - 1) / rows);
}
}  // namespace

// Wavefronts of a workgroup, i.e. 2 kMcWaves - 2 rows: the ring costs (2 NW) /
// (2 NW - 2) of the red solves.  Per pass FP32 256 x 256 / FP64 2048 x 2048 with
// 2, 4 and 8 wavefronts: 11.6 / 9.3 / 11.5 us and 293 / 209 / 244 us; 8 hold
// one workgroup of FP64 per CU, whose loads then overlap with nothing.
constexpr int kMcWaves = 4;

template <typename T>
hipError_t launch_vanka_mc(const SsaArgs<T>& a, T* u_dst, T* v_dst, T* H_dst, T* mask, T* phi_dst,
                           const VankaArgs<T>& vk, hipStream_t st) {
    TimedLaunch tl(std::is_same<T, float>::value ? kTimeVankaMc32 : kTimeVankaMc64, (long)a.ny * a.nx, st);
    constexpr int NW = kMcWaves;
    int gx;
    const int blocks = mc_blocks(a.ny, a.nx, NW, &gx);
    const dim3 b(kRowLanes, NW);
    if (a.P.linear_drag)
        k_mc_pass<T, NW, true><<<blocks, b, 0, st>>>(a, u_dst, v_dst, H_dst, mask, phi_dst, vk, gx);
    else
        k_mc_pass<T, NW, false><<<blocks, b, 0, st>>>(a, u_dst, v_dst, H_dst, mask, phi_dst, vk, gx);
    return hipGetLastError();
}

// Heavy local solves, a nonlinear drag law or five Newton steps and more, are bound
// by instructions, of which the one-launch form has up to 1.5 times as many; it
// wins where its workgroups fit the 256 CUs in as many rounds (fewer launches, less
// traffic), and where the solves are light.  Four passes, one launch / phases, us:
//   linear drag, 3 / 6 / 30 steps      256 x 256: 62/86, 81/104, 229/246;
//     512 x 512: 133/133, 191/167, 658/429;  1024 x 1024: 342/337, 515/422, 1908/1447
//   Weertman drag (m = 1/3), 1 / 3 / 30 steps      256 x 256: 83/104, 149/171, 1036/1065;
//     320 x 320: 138/115, 263/182, 1960/1078;  384 x 384: 145/175, 275/300, 2043/2001;
//     512 x 512: 253/197, 495/328, 3765/2119;  1024 x 1024: 751/583, 1535/1110, 12136/8276
bool mc_phases_faster(int ny, int nx, int newton_steps, bool linear) {
    constexpr long kCus = 256;
    int gx;
    const long one = mc_blocks(ny, nx, kMcWaves, &gx);
    const long phase = (((long)nx + 1) / 2 + kRowLanes - 1) / kRowLanes * (((long)ny + kPhaseRows - 1) / kPhaseRows);
    return (!linear || newton_steps >= 5) && (phase + kCus - 1) / kCus < (one + kCus - 1) / kCus;
}

template <typename T>
hipError_t launch_mc_phases(const SsaArgs<T>& a, T* eta, T* u, T* v, T* H, T* u_alt, T* v_alt, T* H_alt, T* mask,
                            const VankaArgs<T>& vk, hipStream_t st) {
    TimedLaunch tl(std::is_same<T, float>::value ? kTimeVankaMc32 : kTimeVankaMc64, (long)a.ny * a.nx, st);
    k_cell_eta<T><<<dim3((a.nx + 255) / 256, a.ny), 256, 0, st>>>(a, eta);
    const int pairs = (a.nx + 1) / 2;
    const dim3 g((pairs + kRowLanes - 1) / kRowLanes, (a.ny + kPhaseRows - 1) / kPhaseRows), b(kRowLanes, kPhaseRows);
    SsaArgs<T> black = a;
    black.u = u_alt; black.v = v_alt; black.H = H_alt;
    if (a.P.linear_drag) {
        k_mc_phase<T, true><<<g, b, 0, st>>>(a, eta, u_alt, v_alt, H_alt, mask, vk, 0);
        k_mc_phase<T, true><<<g, b, 0, st>>>(black, eta, u, v, H, mask, vk, 1);
    } else {
        k_mc_phase<T, false><<<g, b, 0, st>>>(a, eta, u_alt, v_alt, H_alt, mask, vk, 0);
        k_mc_phase<T, false><<<g, b, 0, st>>>(black, eta, u, v, H, mask, vk, 1);
    }
    return hipGetLastError();
}

// ------------------------------------------------------------ domain tables
namespace {
template <typename T, int NW, bool LINEAR>
__global__ __launch_bounds__(kRowLanes* NW) void k_tab_mc_pass(const TabVankaMc<T>* __restrict__ jobs,
                                                               const int* __restrict__ start, int n) {
    const int e = tab_find(start, n, blockIdx.x);
    const TabVankaMc<T> J = jobs[e];
    const int lb = blockIdx.x - start[e];
    mc_pass_body<T, NW, LINEAR>(lb % J.gx, lb / J.gx, J.a, J.u_dst, J.v_dst, J.H_dst, J.mask, J.phi_dst, J.vk);
}
// wavefronts of a workgroup for a tile setting of 1, 2, 4 or 8
int mc_tile_waves(int rows) { return rows < 2 ? 2 : rows; }
}  // namespace

bool tab_vanka_mc_rows_ok(int rows) { return rows == 1 || rows == 2 || rows == 4 || rows == 8; }
int tab_blocks_vanka_mc(int ny, int nx, int rows, int* gx) { return mc_blocks(ny, nx, mc_tile_waves(rows), gx); }

template <typename T>
hipError_t launch_tab_vanka_mc(const TabVankaMc<T>* jobs, const int* start, int n, int blocks, bool linear, int rows,
                               hipStream_t st) {
    if (n <= 0 || blocks <= 0) return hipSuccess;
    const int nw = mc_tile_waves(rows);
    const dim3 b(kRowLanes, nw);
#define GLIDE_TAB_MC(W)                                                                     \
    if (nw == W) {                                                                          \
        if (linear) k_tab_mc_pass<T, W, true><<<blocks, b, 0, st>>>(jobs, start, n);       \
        else k_tab_mc_pass<T, W, false><<<blocks, b, 0, st>>>(jobs, start, n);             \
        return hipGetLastError();                                                           \
    }
    GLIDE_TAB_MC(2)
    GLIDE_TAB_MC(4)
    GLIDE_TAB_MC(8)
#undef GLIDE_TAB_MC
    return hipErrorInvalidValue;
}

// ------------------------------------------------------------ precision bridge
__global__ __launch_bounds__(256) void k_mixed_batch(MixedBatch b) {
    const MixedJob& q = b.job[blockIdx.y];
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < q.n; k += (long)gridDim.x * blockDim.x) {
        switch (q.op) {
            case kMixTo32:
                static_cast<float*>(q.out)[k] = (float)static_cast<const double*>(q.a)[k];
                break;
            case kMixTo64:
                static_cast<double*>(q.out)[k] = (double)static_cast<const float*>(q.a)[k];
                break;
            case kMixDefect:  // out32 = a32 - (float) b64
                static_cast<float*>(q.out)[k] =
                    static_cast<const float*>(q.a)[k] - (float)static_cast<const double*>(q.b)[k];
                break;
            case kMixUpdate:
            case kMixUpdateH: {  // x64 += y32 - fl32(x64); H: x64 = thk where mask32 is set
                double* x = static_cast<double*>(q.out);
                const double x0 = x[k];
                double xn = x0 + ((double)static_cast<const float*>(q.a)[k] - (double)(float)x0);
                if (q.op == kMixUpdateH && static_cast<const float*>(q.b)[k] > 0.5f) xn = q.val;
                x[k] = xn;
                break;
            }
            case kMixAdd64:  // out64 += (double) a32
                static_cast<double*>(q.out)[k] += (double)static_cast<const float*>(q.a)[k];
                break;
            case kMixNeg32:  // out32 = -(float) a64
                static_cast<float*>(q.out)[k] = -(float)static_cast<const double*>(q.a)[k];
                break;
        }
    }
}

hipError_t launch_mixed_batch(const MixedBatch& b, hipStream_t st) {
    if (b.count <= 0) return hipSuccess;
    long nmax = 0;
    for (int q = 0; q < b.count; ++q) nmax = nmax > b.job[q].n ? nmax : b.job[q].n;
    long bx = (nmax + 255) / 256;
    if (bx > 2048) bx = 2048;
    if (bx < 1) bx = 1;
    k_mixed_batch<<<dim3((unsigned)bx, b.count), 256, 0, st>>>(b);
    return hipGetLastError();
}

// ------------------------------------------------------------ Krylov helpers
// The flexible GMRES outer iteration of the mixed adjoint solve works on flat
// FP64 vectors (the u, v and H multipliers of a level one after another);
// these are its inner products and updates.  The sums are formed in a fixed
// order (fixed grid, fixed block reduction), so repeated solves are bitwise
// identical.

// partial[q * gridDim.x + b]: block b's part of <w, V_q> for q < nq (V_q at
// V + q * ld), and of <w, w> at q = nq.
__global__ __launch_bounds__(256) void k_krylov_dots(const double* __restrict__ w, const double* __restrict__ V,
                                                     long ld, long n, int nq, double* __restrict__ partial) {
    __shared__ double red[4][kKrylovMaxDots + 1];
    double acc[kKrylovMaxDots + 1];
#pragma unroll
    for (int q = 0; q <= kKrylovMaxDots; ++q) acc[q] = 0.0;
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x) {
        const double wk = w[k];
#pragma unroll
        for (int q = 0; q < kKrylovMaxDots; ++q)
            if (q < nq) acc[q] = fma(wk, V[q * ld + k], acc[q]);
        acc[kKrylovMaxDots] = fma(wk, wk, acc[kKrylovMaxDots]);
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q <= kKrylovMaxDots; ++q) {
        if (q < nq || q == kKrylovMaxDots) {
            double v = acc[q];
            for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
            if (lane == 0) red[wv][q] = v;
        }
    }
    __syncthreads();
    if (threadIdx.x <= nq) {
        const int q = threadIdx.x == nq ? kKrylovMaxDots : threadIdx.x;
        partial[(long)threadIdx.x * gridDim.x + blockIdx.x] = (red[0][q] + red[1][q]) + (red[2][q] + red[3][q]);
    }
}

// out[q] = sum over the nb partials of q, q <= nq (one block per q).
__global__ __launch_bounds__(256) void k_krylov_reduce(const double* __restrict__ partial, int nb,
                                                       double* __restrict__ out) {
    __shared__ double red[4];
    double v = 0.0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) v += partial[(long)blockIdx.x * nb + b];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// out[k] += sign * sum_{q < nq} c[q] V[q * ld + k]  (c on the device).
__global__ __launch_bounds__(256) void k_krylov_axpy(double* __restrict__ out, const double* __restrict__ V, long ld,
                                                     long n, int nq, const double* __restrict__ c, double sign) {
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int q = 0; q < nq; ++q) s = fma(c[q], V[q * ld + k], s);
        out[k] = fma(sign, s, out[k]);
    }
}

hipError_t launch_krylov_dots(const double* w, const double* V, long ld, long n, int nq, double* partial,
                              double* out, hipStream_t st) {
    if (nq < 0 || nq > kKrylovMaxDots) return hipErrorInvalidValue;
    k_krylov_dots<<<kKrylovBlocks, 256, 0, st>>>(w, V, ld, n, nq, partial);
    k_krylov_reduce<<<nq + 1, 256, 0, st>>>(partial, kKrylovBlocks, out);
    return hipGetLastError();
}

hipError_t launch_krylov_axpy(double* out, const double* V, long ld, long n, int nq, const double* c, double sign,
                              hipStream_t st) {
    if (nq <= 0 || n <= 0) return hipSuccess;
    long b = (n + 255) / 256;
    if (b > 2048) b = 2048;
    k_krylov_axpy<<<(unsigned)b, 256, 0, st>>>(out, V, ld, n, nq, c, sign);
    return hipGetLastError();
}

#define GLIDE_MC_INSTANTIATE(T)                                                                                     \
    template hipError_t launch_pin_rows<T>(T*, T*, T*, const T*, int, int, hipStream_t);                           \
    template hipError_t launch_vanka_mc<T>(const SsaArgs<T>&, T*, T*, T*, T*, T*, const VankaArgs<T>&, hipStream_t); \
    template hipError_t launch_mc_phases<T>(const SsaArgs<T>&, T*, T*, T*, T*, T*, T*, T*, T*, const VankaArgs<T>&, \
                                            hipStream_t);

GLIDE_MC_INSTANTIATE(double)
GLIDE_MC_INSTANTIATE(float)

#define GLIDE_MC_TAB_INSTANTIATE(T)                                                                                 \
    template hipError_t launch_tab_vanka_mc<T>(const TabVankaMc<T>*, const int*, int, int, bool, int, hipStream_t);

GLIDE_MC_TAB_INSTANTIATE(double)
GLIDE_MC_TAB_INSTANTIATE(float)

}  // namespace glide
