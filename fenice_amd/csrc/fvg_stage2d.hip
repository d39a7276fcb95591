// One Runge-Kutta stage of a 2-D mesh (FP64 fluxes, midpoint quadrature, reconstructed faces) in one launch: primitives
// with their halo, viscous gradients, x and y fluxes, divergence and stage combination, tile by tile in LDS. The same
// operations in the same order as k_cells, k_faces and k_update, so the same bits.
//
// A small mesh is bound by the latency of a chain of launches (64^2 viscous cavity: four passes of 6-16 us a stage); a
// large one by FP64 arithmetic in the face passes and by HBM in the two others, which move primitives, gradients and
// fluxes (2048^2: 48 and 120 us of 491 a stage). Here a block of 512 threads takes 15 x 15 cells: 21 x 21 primitives and
// 17 x 17 gradients, one per thread, then 16 x 15 x faces on the lower half of the block while the upper half takes the
// 15 x 16 y faces. It repeats 1/15 of the faces. Two blocks are resident on a CU (four wavefronts per SIMD, the
// registers' limit), so one block's loads run under the other's arithmetic.
// A stage never writes its own input (neighbouring tiles still read it): the first stage stores its residual, since
// its step size is not known before every tile is done. The second SSP-RK3 stage forms the first one's result, U + dt R,
// as it loads it (KP::R0) instead of reading what a pass of its own stored (a step of the 64^2 cavity 81 -> 77 us, of
// 2048^2 1,340 -> 1,294).
// Measured per step (SSP-RK3): viscous MUSCL cavity 32^2 125 -> 81 us, 64^2 118 -> 79, 400^2 170 -> 132; periodic WENO5-Z
// 100 x 90 70 -> 44 us, 511 x 700 206 -> 159, 2048^2 1,798 -> 1,353.
#define FVG_SUMMED_INPUT
#include "fvg_kernels_impl.hpp"

namespace fvg {

namespace {

constexpr int TC = kStageTile;        // cells of a tile per side
constexpr int TW = TC + 2 * PH;       // cells with primitives
constexpr int TG = TC + 2;            // cells with gradients
static_assert(TW * TW <= 512 && TG * TG <= 512 && (TC + 1) * TC <= 256, "thread assignments of k_stage2d");

template <bool VISC> struct StageTile {
    double W[4][TW][TW];
    double Fx[4][TC][TC + 1], Fy[4][TC + 1][TC];
    int wide[8];
};
template <> struct StageTile<true> {
    double W[4][TW][TW];
    double Fx[4][TC][TC + 1], Fy[4][TC + 1][TC];
    int wide[8];
    double G[4][TG][TG];
    double Vx[3][TC][TC + 1], Vy[3][TC + 1][TC];
};

// Where the primitives at coordinate g of an axis come from (push_halo): the coordinate of the source cell, with
// ghost set when its ghost state beyond side 2 d + hi is taken; false when no stencil reads them.
template <bool PER>
__device__ __forceinline__ bool source_of(const KP& p, int d, int g, int& src, bool& ghost) {
    const int n = ncell(p, d);
    src = g;
    if (g >= 0 && g < n) return true;
    if (g < -PH || g >= n + PH) return false;
    const bool hi = g >= n;
    const int h = PER ? 1 : halo_of(p, 2 * d + hi);
    if (h == 1) {
        src = hi ? (g - n) % n : n - 1 - (-1 - g) % n;
    } else if (h == 2) {
        src = hi ? 2 * n - 1 - g : -1 - g;
        ghost = true;
        return src >= 0 && src < n;
    } else {
        src = hi ? n - 1 : 0;
    }
    return true;
}

// the viscous flux of face (i, j) normal to D (viscous_face in 2-D, from the tile): (fi, fj) its place in the tile
template <int D, bool IR, bool PER>
__device__ __forceinline__ void tile_viscous(const KP& p, const StageTile<true>& s, int i, int j, int fi, int fj, double* out) {
    const int t = D == 0 ? i : j, n = ncell(p, D);
    const bool lo = t == 0, hi = t == n, pad = !PER && !wrap_of(p, D);
    double vL[2], vR[2], TL, TR, w[4];
    auto tile_prim = [&](int x, int y) {
#pragma unroll
        for (int q = 0; q < 4; ++q) w[q] = s.W[q][y][x];
    };
    if (pad && lo) visc_pad_prim<4>(p, D == 0 ? -1 : i, D == 1 ? -1 : j, 0, w);
    else tile_prim(fi + PH - (D == 0), fj + PH - (D == 1));
    vL[0] = w[1], vL[1] = w[2];
    TL = dvp<IR>(w[3], w[0]);
    if (pad && hi) visc_pad_prim<4>(p, D == 0 ? n : i, D == 1 ? n : j, 0, w);
    else tile_prim(fi + PH, fj + PH);
    vR[0] = w[1], vR[1] = w[2];
    TR = dvp<IR>(w[3], w[0]);
    const bool phys = !PER && p.bo2 && !vper_of(p, D) && (lo || hi);
    const int tg = lo ? -1 : n, tc = lo ? 0 : n - 1;
    constexpr int B = 1 - D;   // the tangential axis; d u_B / d x_B and d u_D / d x_B
    double own, nor;
    if (phys) {
        double d[2];
        boundary_cross<4, D>(p, i, j, 0, tg, tc, B, d);
        own = d[B];
        nor = d[D];
    } else {   // the gradients of the cells on both sides of the face
        const int xl = fi + (D == 1), yl = fj + (D == 0);
        own = 0.5 * (s.G[B * 2 + B][yl][xl] + s.G[B * 2 + B][fj + 1][fi + 1]);
        nor = 0.5 * (s.G[D * 2 + B][yl][xl] + s.G[D * 2 + B][fj + 1][fi + 1]);
    }
    const double h = hstep(p, D), inv_h = inv_hstep(p, D), mu = p.mu, kc = p.k_cond;
    const double u_f = 0.5 * (vL[0] + vR[0]), v_f = 0.5 * (vL[1] + vR[1]);
    const double du = by_const<IR>(vR[0] - vL[0], h, inv_h), dvel = by_const<IR>(vR[1] - vL[1], h, inv_h), dT = by_const<IR>(TR - TL, h, inv_h);
    if constexpr (D == 0) {
        const double du_dy = nor, dv_dy = own;
        const double tau_xx = mu * (MU_DIAG * du - MU_OFF * dv_dy), tau_xy = mu * (du_dy + dvel), q_x = -kc * dT, ar = p.dy;
        out[0] = tau_xx * ar;
        out[1] = tau_xy * ar;
        out[2] = (u_f * tau_xx + v_f * tau_xy - q_x) * ar;
    } else {
        const double du_dx = own, dv_dx = nor;
        const double tau_yy = mu * (MU_DIAG * dvel - MU_OFF * du_dx), tau_yx = mu * (du + dv_dx), q_y = -kc * dT, ar = p.dx;
        out[0] = tau_yx * ar;
        out[1] = tau_yy * ar;
        out[2] = (u_f * tau_yx + v_f * tau_yy - q_y) * ar;
    }
}

// face (i, j) normal to D: states (face_states from the tile), Riemann flux, viscous flux; returns its wave speed
template <int D, int RECON, bool VISC, bool IR, bool PER>
__device__ __forceinline__ double tile_face(const KP& p, StageTile<VISC>& s, int i, int j, int fi, int fj) {
    const int t = D == 0 ? i : j, n = ncell(p, D);
    const bool lo = t == 0, hi = t == n;
    double UL[4], UR[4], F[4], sm;
    if (PER || (t > 0 && t < n) || (lo && halo_of(p, 2 * D)) || (hi && halo_of(p, 2 * D + 1))) {
        double wl[4], wr[4];
        const double we = p.weno_eps;
        auto cell = [&](int q, int k) {   // cell t - 3 + k of the face's line
            return D == 0 ? s.W[q][fj + PH][fi + k] : s.W[q][fj + k][fi + PH];
        };
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if constexpr (RECON == 3) {
                const double c0 = cell(q, 0), c1 = cell(q, 1), c2 = cell(q, 2), c3 = cell(q, 3), c4 = cell(q, 4), c5 = cell(q, 5);
                wl[q] = weno5z<double, IR>(c0, c1, c2, c3, c4, we);
                wr[q] = weno5z<double, IR>(c5, c4, c3, c2, c1, we);
            } else {
                const double c1 = cell(q, 1), c2 = cell(q, 2), c3 = cell(q, 3), c4 = cell(q, 4);
                if constexpr (RECON == 2) {
                    wl[q] = weno3z<double, IR>(c1, c2, c3, we);
                    wr[q] = weno3z<double, IR>(c4, c3, c2, we);
                } else {
                    wl[q] = muscl_wl<IR>(p.lim, c1, c2, c3);
                    wr[q] = muscl_wr<IR>(p.lim, c2, c3, c4);
                }
            }
        }
        p2c<4, IR>(p.rs.eos, wl, UL);
        p2c<4, IR>(p.rs.eos, wr, UR);
    } else {   // a side without a halo: the first-order states
        const int il = D == 0 ? t - 1 : i, jl = D == 1 ? t - 1 : j;
        if (!lo) load_cons<4>(p, cidx(p, il, jl, 0), UL);
        else outside_first_order<4>(p, D, 2 * D, i, j, 0, UL);
        if (!hi) load_cons<4>(p, cidx(p, i, j, 0), UR);
        else outside_first_order<4>(p, D, 2 * D + 1, il, jl, 0, UR);
        roundtrip<4>(p.rs.eos, UL);
        roundtrip<4>(p.rs.eos, UR);
    }
    face_flux<4, IR>(p.rs, UL, UR, D, F, sm);
#pragma unroll
    for (int q = 0; q < 4; ++q) (D == 0 ? s.Fx[q][fj][fi] : s.Fy[q][fj][fi]) = F[q];
    if constexpr (VISC) {
        double v[3];
        tile_viscous<D, IR, PER>(p, s, i, j, fi, fj, v);
#pragma unroll
        for (int q = 0; q < 3; ++q) (D == 0 ? s.Vx[q][fj][fi] : s.Vy[q][fj][fi]) = v[q];
    }
    return sm;
}

template <int RECON, bool VISC, bool IR, bool PER>
__device__ __forceinline__ double tile_faces(const KP& p, StageTile<VISC>& s, int i0, int j0) {
    const int h = threadIdx.x & 255;
    if (threadIdx.x < 256) {
        const int fi = h % (TC + 1), fj = h / (TC + 1);
        if (fj < TC && i0 + fi <= p.nx && j0 + fj < p.ny) return tile_face<0, RECON, VISC, IR, PER>(p, s, i0 + fi, j0 + fj, fi, fj);
    } else {
        const int fi = h % TC, fj = h / TC;
        if (fj <= TC && i0 + fi < p.nx && j0 + fj <= p.ny) return tile_face<1, RECON, VISC, IR, PER>(p, s, i0 + fi, j0 + fj, fi, fj);
    }
    return 0.0;
}

}   // namespace

template <int RECON, bool VISC, bool PER>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void k_stage2d(KP p, int upd, const double* U0, const double* Ut, double* out) {
    __shared__ StageTile<VISC> s;
    const int t = threadIdx.x, i0 = blockIdx.x * TC, j0 = blockIdx.y * TC;
    // primitives of the tile and its halo; the corners of the halo are read by no stencil
    bool wide = false, have = false, gx = false, gy = false;
    const int wi = t % TW, wj = t / TW, gi = i0 - PH + wi, gj = j0 - PH + wj;
    int si = 0, sj = 0;
    double u[4];
    if (t < TW * TW) {
        const bool ox = gi < 0 || gi >= p.nx, oy = gj < 0 || gj >= p.ny;
        have = !(ox && oy) && source_of<PER>(p, 0, gi, si, gx) && source_of<PER>(p, 1, gj, sj, gy);
        if (have) load_cons<4>(p, cidx(p, si, sj, 0), u);
    }
    if (p.st->done) return;   // uniform; read behind the loads
    if (have) {
        double w[4];
        if (!PER && (gx || gy)) {
            double ug[4];
            ghost_state<4>(p.rs.eos, p.bp, gx ? (gi < 0 ? 0 : 1) : (gj < 0 ? 2 : 3), u, ug);
            c2p<4>(p.rs.eos, ug, w, (double*)nullptr);
        } else {
            c2p<4>(p.rs.eos, u, w, (double*)nullptr);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            s.W[q][wj][wi] = w[q];
            wide |= !value_in_range(w[q]);
        }
    }
    double bound = 0.0, local = 0.0;
    if constexpr (VISC) {
        // gradients of the tile and the cells around it: beyond a side, of the opposite cell on a periodic axis (that
        // is what a seam face takes) and of the edge cell on the others
        const int ti = t % TG, tj = t / TG;
        int ci = i0 - 1 + ti, cj = j0 - 1 + tj;
        if (t < TG * TG && ci <= p.nx && cj <= p.ny) {
            ci = ci < 0 ? (PER || p.vper[0] ? p.nx - 1 : 0) : (ci >= p.nx ? (PER || p.vper[0] ? 0 : p.nx - 1) : ci);
            cj = cj < 0 ? (PER || p.vper[1] ? p.ny - 1 : 0) : (cj >= p.ny ? (PER || p.vper[1] ? 0 : p.ny - 1) : cj);
            double d[2][3], v[4], w[4], G[2][2];
            load_cons<4>(p, cidx(p, ci, cj, 0), v);
            cell_differences<4, PER, double>(p, ci, cj, 0, d);
            c2p<4>(p.rs.eos, v, w, (double*)nullptr);
            if (!p.ir || !cell_gradients_f64<4, true>(p, d, w, G, bound)) cell_gradients_f64<4, false>(p, d, w, G, bound);
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b) s.G[a * 2 + b][tj][ti] = G[a][b];
        }
    }
    const bool any = __any(wide);
    if ((t & 63) == 0) s.wide[t >> 6] = any;
    __syncthreads();
    int nwide = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) nwide |= s.wide[k];
    double speed;
    if (p.ir != 0 && __builtin_amdgcn_readfirstlane(nwide) == 0) speed = tile_faces<RECON, VISC, true, PER>(p, s, i0, j0);
    else speed = tile_faces<RECON, VISC, false, PER>(p, s, i0, j0);
    if (speed > local) local = speed;
    __syncthreads();
    const int x = t % TC, y = t / TC, i = i0 + x, j = j0 + y;
    if (t < TC * TC && i < p.nx && j < p.ny) {
        const long long c = cidx(p, i, j, 0);
        double R[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double fl = s.Fx[q][y][x], fr = s.Fx[q][y][x + 1], fb = s.Fy[q][y][x], ft = s.Fy[q][y + 1][x];
            R[q] = ((0.0 - (fr * p.Ax - fl * p.Ax)) - (ft * p.Ay - fb * p.Ay)) * p.inv_vol;
        }
        if constexpr (VISC) {
            R[0] = R[0] + 0.0;   // the zero viscous flux of the density slot
#pragma unroll
            for (int q = 1; q < 4; ++q) {
                const double fl = s.Vx[q - 1][y][x], fr = s.Vx[q - 1][y][x + 1], fb = s.Vy[q - 1][y][x], ft = s.Vy[q - 1][y + 1][x];
                R[q] = R[q] + ((0.0 + (fr - fl)) + (ft - fb)) * p.inv_vol;
            }
        }
        switch (upd) {   // uniform
        case UPD_RESIDUAL: combine<4, UPD_RESIDUAL>(p, c, R, U0, Ut, out); break;
        case UPD_RK2_2: combine<4, UPD_RK2_2>(p, c, R, U0, Ut, out); break;
        case UPD_RK3_2:
            if (p.R0) {   // Ut = U + dt R0 as load_cons makes it
                const double dt = p.st->dt;
                double ut[4];
                load_cons<4>(p, c, ut);
#pragma unroll
                for (int q = 0; q < 4; ++q) out[q * p.nc + c] = 0.75 * U0[q * p.nc + c] + 0.25 * (ut[q] + dt * R[q]);
            } else {
                combine<4, UPD_RK3_2>(p, c, R, U0, Ut, out);
            }
            break;
        default: combine<4, UPD_RK3_3>(p, c, R, U0, Ut, out); break;
        }
    }
    const size_t slot = (blockIdx.y * gridDim.x + blockIdx.x) % kSpeedSlots;
    block_max_to(local, p.spd + ((size_t)SPD_CONV * kSpeedSlots + slot) * kSlotStride);
    if constexpr (VISC) {
        __syncthreads();   // block_max_to's LDS
        block_max_to(bound, p.spd + ((size_t)SPD_VISC * kSpeedSlots + slot) * kSlotStride);
    }
}

#define FVG_STAGE2D(R)                                                                          \
    template __global__ void k_stage2d<R, false, false>(KP, int, const double*, const double*, double*); \
    template __global__ void k_stage2d<R, false, true>(KP, int, const double*, const double*, double*);  \
    template __global__ void k_stage2d<R, true, false>(KP, int, const double*, const double*, double*);  \
    template __global__ void k_stage2d<R, true, true>(KP, int, const double*, const double*, double*);
FVG_STAGE2D(1)
FVG_STAGE2D(2)
FVG_STAGE2D(3)

}   // namespace fvg
