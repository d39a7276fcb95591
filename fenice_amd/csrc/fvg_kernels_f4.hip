// flux_quadrature = fourth on the device (FP64, the reference's bits): fourth_order_fluxes and the conserved
// reconstruction it takes (Schemes.cpp:1210-1349, 1954-2134), as three passes over the faces of one axis at a time.
//
//   k4_states<D>  WENO3-Z / WENO5-Z of the padded conservative state Wc at every face with a full stencil, the
//                 admissibility check (positive states inside the widened range of the stencil cells, else the two
//                 cells next to the face); a face without a full stencil takes its first-order boundary state as
//                 it is. Flags the faces that are good: a full stencil, both states positive, the shock sensor quiet.
//   k4_points<D>  point values A = U - (0 + sum over the transverse axes of (U[+1] - 2 U + U[-1])) / 24 where the
//                 face and its transverse neighbours are good and A stays positive (flag pt), then the Riemann flux
//                 Fp of the point values (of the averages elsewhere); its block maxima give the wave speed.
//   k4_fluxes<D>  F = Fp + (0 + sum of (Fp[+1] - 2 Fp + Fp[-1])) / 24 where the face and its transverse
//                 neighbours have point values, the flux of the averaged states where only the face has, else Fp;
//                 stored with the viscous face flux for k_update, as k_faces stores its fluxes.
//
// Transverse neighbours are faces of the same axis one lattice step away; across a periodic axis they wrap to the
// other side (the reference's `periodic`: both sides of the axis periodic, whatever its halo), else the face has no
// correction. The three passes exchange the face states, flags and fluxes through q4_* buffers sized for the
// largest axis and reused axis after axis.
#include "fvg_kernels_impl.hpp"

namespace fvg {

namespace {

// p > 0 and rho > 0 without a division, and the pressure (Schemes.cpp:1241-1243, 1287, 1966-1969). With NV = 4
// the absent rho w adds +0 to |m|^2, which leaves it as it is.
template <int NV> __device__ __forceinline__ double q4_m2(const double* u) {
    double m = u[1] * u[1] + u[2] * u[2];
    if constexpr (NV == 5) m = m + u[4] * u[4];
    return m;
}
template <int NV> __device__ __forceinline__ bool q4_positive(double g1, double gp, const double* u) {
    return u[0] > 0.0 && g1 * (u[3] * u[0] - 0.5 * q4_m2<NV>(u)) > gp * u[0];
}
template <int NV, bool IR = false> __device__ __forceinline__ double q4_pressure(double g1, double gp, const double* u) {
    return g1 * (u[3] - dvx<IR>(0.5 * q4_m2<NV>(u), u[0])) - gp;
}

// the face one lattice step s (-1, +1) from face f along transverse axis t, -1 when there is none
// (fourth_order_fluxes' nbr, Schemes.cpp:2022-2027)
template <int D>
__device__ __forceinline__ long long q4_nbr(const KP& p, long long f, int ct, int t, int s) {
    const long long ni = p.nx + (D == 0), nj = p.ny + (D == 1);
    const long long st = t == 0 ? 1 : (t == 1 ? ni : ni * nj);
    const int n = ncell(p, t);
    const int c = ct + s;
    if (c >= 0 && c < n) return f + s * st;
    if (!vper_of(p, t)) return -1;
    return f - s * (long long)(n - 1) * st;
}

// the transverse axes of the faces normal to D, in increasing order
template <int NV, int D> struct Trans {
    static constexpr int n = NV - 3;   // 1 in 2-D, 2 in 3-D
    static constexpr int t0 = D == 0 ? 1 : 0;
    static constexpr int t1 = D == 2 ? 1 : 2;
};

// the transverse neighbours of face f (f itself where there is none), and whether all are there and flagged as f is. All
// flags are read at once: a chain of reads, each waiting for the flag before it, is what these short passes would wait for.
template <int NV, int D>
__device__ __forceinline__ bool q4_neighbours(const KP& p, const unsigned char* flag, long long f, int i, int j, int k, long long (*nb)[2]) {
    using TR = Trans<NV, D>;
    const int ct[2] = {coord(TR::t0, i, j, k), coord(TR::t1, i, j, k)};
    int ok = flag[f];
#pragma unroll
    for (int u = 0; u < TR::n; ++u)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const long long x = q4_nbr<D>(p, f, ct[u], u ? TR::t1 : TR::t0, 2 * s - 1);
            nb[u][s] = x < 0 ? f : x;
            ok &= int(x >= 0) & int(flag[nb[u][s]]);
        }
    return ok != 0;
}

template <int NV>
__device__ __forceinline__ void q4_load(const double* planes, long long n, long long f, double* u) {
#pragma unroll
    for (int q = 0; q < NV; ++q) u[q] = planes[q * n + f];
}

}   // namespace

// R: the reconstruction, 2 WENO3-Z (four cells t-2 .. t+1), 3 WENO5-Z (six cells t-3 .. t+2)
// IR: the operands are in range (every value of Wc in value_in_range)
template <int NV, int D, int R, bool IR>
__device__ __forceinline__ void k4_states_face(const KP& p, long long f) {
    int i, j, k, t;
    face_coords<NV, D>(p, f, i, j, k, t);
    const int n = ncell(p, D);
    const bool lo = t == 0, hi = t == n;
    const bool upgrade = (t > 0 && t < n) || (lo && halo_of(p, 2 * D)) || (hi && halo_of(p, 2 * D + 1));
    const double g1 = p.rs.eos.gamma - 1.0, gp = p.rs.eos.stiff ? p.rs.eos.gamma * p.rs.eos.p_inf : 0.0;
    double ul[NV], ur[NV];
    if (upgrade) {
        const double we = p.weno_eps;
        constexpr int NS = R == 3 ? 6 : 4;
        double c[NS][NV];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const long long pc = pidx_d(p, D, i, j, k, t - NS / 2 + s);
#pragma unroll
            for (int q = 0; q < NV; ++q) c[s][q] = p.Wc[q * p.npad + pc];
        }
        if constexpr (R == 3) {
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                ul[q] = weno5z<double, IR>(c[0][q], c[1][q], c[2][q], c[3][q], c[4][q], we);
                ur[q] = weno5z<double, IR>(c[5][q], c[4][q], c[3][q], c[2][q], c[1][q], we);
            }
        } else {
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                ul[q] = weno3z<double, IR>(c[0][q], c[1][q], c[2][q], we);
                ur[q] = weno3z<double, IR>(c[3][q], c[2][q], c[1][q], we);
            }
        }
        // admissible: positive, and the density and pressure inside the range of the stencil cells widened by the
        // range's own width (ConservedLines::line, Schemes.cpp:1288-1318)
        bool ok = q4_positive<NV>(g1, gp, ul) && q4_positive<NV>(g1, gp, ur);
        if (ok) {
            double rlo = 1e300, rhi = -1e300, plo = 1e300, phi = -1e300;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const double pc = q4_pressure<NV, IR>(g1, gp, c[s]);
                rlo = smin(rlo, c[s][0]);
                rhi = smax(rhi, c[s][0]);
                plo = smin(plo, pc);
                phi = smax(phi, pc);
            }
            const double rw = rhi - rlo, pw = phi - plo;
            rlo -= rw;
            rhi += rw;
            plo -= pw;
            phi += pw;
            const double pl = q4_pressure<NV, IR>(g1, gp, ul), pr = q4_pressure<NV, IR>(g1, gp, ur);
            ok = ul[0] >= rlo && ul[0] <= rhi && pl >= plo && pl <= phi;
            ok = ok && ur[0] >= rlo && ur[0] <= rhi && pr >= plo && pr <= phi;
        }
        if (!ok) {   // the cells on both sides: stencil positions 2, 3 of the six, 1, 2 of the four
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                ul[q] = c[NS / 2 - 1][q];
                ur[q] = c[NS / 2][q];
            }
        }
    } else {   // a side without a halo: the first-order boundary states, not converted
        const int il = D == 0 ? t - 1 : i, jl = D == 1 ? t - 1 : j, kl = D == 2 ? t - 1 : k;
        if (!lo) load_cons<NV>(p, cidx(p, il, jl, kl), ul);
        else outside_first_order<NV>(p, D, 2 * D, i, j, k, ul);
        if (!hi) load_cons<NV>(p, cidx(p, i, j, k), ur);
        else outside_first_order<NV>(p, D, 2 * D + 1, il, jl, kl, ur);
    }
    // good: a full stencil, positive states, the shock sensor quiet (Schemes.cpp:1987-2005)
    bool good = upgrade && q4_positive<NV>(g1, gp, ul) && q4_positive<NV>(g1, gp, ur);
    if (good && p.rs.blend > 0.0) {
        const double pL = q4_pressure<NV, IR>(g1, gp, ul), pR = q4_pressure<NV, IR>(g1, gp, ur);
        if (fabs(pR - pL) > p.rs.blend * smin(pL, pR)) good = false;
    }
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        p.q4_UL[q * p.q4_n + f] = ul[q];
        p.q4_UR[q * p.q4_n + f] = ur[q];
    }
    p.q4_good[f] = good ? 1 : 0;
}

template <int NV, int D, int R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k4_states(KP p) {
    const long long f = xcd_block() * blockDim.x + threadIdx.x;
    if (f >= p.nfa[D] || p.st->done) return;
    if (in_range(p)) k4_states_face<NV, D, R, true>(p, f);
    else k4_states_face<NV, D, R, false>(p, f);
}

template <int NV, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k4_points(KP p) {
    using TR = Trans<NV, D>;
    const long long f = xcd_block() * blockDim.x + threadIdx.x;
    double local = 0.0;
    if (f < p.nfa[D] && !p.st->done) {
        int i, j, k, t;
        face_coords<NV, D>(p, f, i, j, k, t);
        double al[NV], ar[NV];
        q4_load<NV>(p.q4_UL, p.q4_n, f, al);
        q4_load<NV>(p.q4_UR, p.q4_n, f, ar);
        bool pt = false;
        {
            long long nb[2][2];
            if (q4_neighbours<NV, D>(p, p.q4_good, f, i, j, k, nb)) {
                double pl[NV], pr[NV];
#pragma unroll
                for (int q = 0; q < NV; ++q) {
                    const double* L = p.q4_UL + q * p.q4_n;
                    const double* R = p.q4_UR + q * p.q4_n;
                    double dl = 0.0, dr = 0.0;
#pragma unroll
                    for (int u = 0; u < TR::n; ++u) {
                        dl += L[nb[u][1]] - 2.0 * al[q] + L[nb[u][0]];
                        dr += R[nb[u][1]] - 2.0 * ar[q] + R[nb[u][0]];
                    }
                    pl[q] = al[q] - dl / 24.0;
                    pr[q] = ar[q] - dr / 24.0;
                }
                const double g1 = p.rs.eos.gamma - 1.0, gp = p.rs.eos.stiff ? p.rs.eos.gamma * p.rs.eos.p_inf : 0.0;
                if (q4_positive<NV>(g1, gp, pl) && q4_positive<NV>(g1, gp, pr)) {
#pragma unroll
                    for (int q = 0; q < NV; ++q) {
                        al[q] = pl[q];
                        ar[q] = pr[q];
                    }
                    pt = true;
                }
            }
        }
        double F[NV], sm;
        face_flux<NV>(p.rs, al, ar, D, F, sm);
        if (sm > local) local = sm;
#pragma unroll
        for (int q = 0; q < NV; ++q) p.q4_Fp[q * p.q4_n + f] = F[q];
        p.q4_pt[f] = pt ? 1 : 0;
    }
    block_max_slot(p, local, SPD_CONV);
}

// the corrected flux of face f
template <int NV, int D>
__device__ __forceinline__ void q4_flux(const KP& p, long long f, int i, int j, int k, double* F) {
    using TR = Trans<NV, D>;
    q4_load<NV>(p.q4_Fp, p.q4_n, f, F);
    long long nb[2][2];
    const bool pt = p.q4_pt[f] != 0, full = q4_neighbours<NV, D>(p, p.q4_pt, f, i, j, k, nb);
    double C[NV];   // of the neighbours' fluxes, read with the flags
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        const double* P = p.q4_Fp + q * p.q4_n;
        double d = 0.0;
#pragma unroll
        for (int u = 0; u < TR::n; ++u) d += P[nb[u][1]] - 2.0 * F[q] + P[nb[u][0]];
        C[q] = d;
    }
    if (pt) {
        if (full) {
#pragma unroll
            for (int q = 0; q < NV; ++q) F[q] = F[q] + C[q] / 24.0;
        } else {   // a point value without the full correction: the flux of the averaged states
            double ul[NV], ur[NV], sm;
            q4_load<NV>(p.q4_UL, p.q4_n, f, ul);
            q4_load<NV>(p.q4_UR, p.q4_n, f, ur);
            face_flux<NV>(p.rs, ul, ur, D, F, sm);
        }
    }
}

// PER as in k_faces: the viscous face flux without boundary code
template <int NV, int D, bool PER>
__global__ __launch_bounds__(256) void k4_fluxes(KP p) {
    const long long f = xcd_block() * blockDim.x + threadIdx.x;
    if (f >= p.nfa[D] || p.st->done) return;
    int i, j, k, t;
    face_coords<NV, D>(p, f, i, j, k, t);
    double F[NV];
    q4_flux<NV, D>(p, f, i, j, k, F);
    if (in_range(p)) store_face<NV, D, double, true, PER>(p, f, i, j, k, t, ncell(p, D), F);
    else store_face<NV, D, double, false, PER>(p, f, i, j, k, t, ncell(p, D), F);
}

// the x faces' k4_fluxes with the update, after the other axes (k_xlast). 96^3, a stage's corrected fluxes and update: 153 +
// 68 -> 177 us, and 7 of the first stage's k_axpy; reading the flags at once (q4_neighbours) is 2 of it and 2 of k4_points.
template <bool PER>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k4_xlast(KP p, int upd, const double* __restrict__ U0,
                                                                                       const double* __restrict__ Ut, double* __restrict__ out) {
    if (p.st->done) return;   // uniform: the whole grid leaves
    const int lane = threadIdx.x & 63;
    const long long f = (xcd_block() * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 63 + lane;
    const bool active = f < p.nfa[0];
    int i = 0, j = 0, k = 0, t;
    double F[5] = {}, Fv[4] = {};
    if (active) {
        face_coords<5, 0>(p, f, i, j, k, t);
        q4_flux<5, 0>(p, f, i, j, k, F);
        if (p.viscous) {
            if (in_range(p)) viscous_face<5, 0, double, true, PER>(p, i, j, k, i, p.nx, Fv);
            else viscous_face<5, 0, double, false, PER>(p, i, j, k, i, p.nx, Fv);
        }
    }
    xlast_cell<double>(p, active, lane, i, j, k, F, Fv, upd, U0, Ut, out);
}


#define FVG_INST_Q4(NV, D)                              \
    template __global__ void k4_states<NV, D, 2>(KP); \
    template __global__ void k4_states<NV, D, 3>(KP); \
    template __global__ void k4_points<NV, D>(KP);

#define FVG_INST_Q4F(NV, D)                              \
    template __global__ void k4_fluxes<NV, D, true>(KP); \
    template __global__ void k4_fluxes<NV, D, false>(KP);
FVG_INST_Q4(4, 0)
FVG_INST_Q4(4, 1)
FVG_INST_Q4(5, 0)
FVG_INST_Q4(5, 1)
FVG_INST_Q4(5, 2)
FVG_INST_Q4F(4, 0)
FVG_INST_Q4F(4, 1)
FVG_INST_Q4F(5, 1)
FVG_INST_Q4F(5, 2)
template __global__ void k4_xlast<true>(KP, int, const double*, const double*, double*);
template __global__ void k4_xlast<false>(KP, int, const double*, const double*, double*);

}   // namespace fvg
