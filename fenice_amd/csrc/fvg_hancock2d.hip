// One MUSCL-Hancock step of a periodic, inviscid 2-D mesh in one launch: primitives, limited and advanced states, x and y
// fluxes, divergence and update, tile by tile in LDS (Schemes.cpp:2135-2199, 2907-3016; TimeScheme.cpp:285-319).
//
// What bounds such a step is latency: at 256^2 the separate passes (k_cells, k_hancock, two face passes, k_update) take
// 3.5-7 us each, a chain of five memory round trips, for 65,536 cells that the chip computes in under 2 us; on a large
// mesh they move the states (128 B a cell), fluxes and primitives through HBM. Here a block of 512 threads takes a
// tile of 14 x 14 cells: 18 x 18 primitives, 16 x 16 cells of advanced states (one per thread of the lower half), then
// 15 x 14 x faces on the lower half while the upper half takes 14 x 15 y faces. A tile repeats (16/14)^2 of the predictor
// and 15/14 of the face work; 12 x 12 would repeat 1.78 of the predictor, 30 x 14 leaves 171 tiles at 256^2, fewer than
// the chip has CUs. Neighbouring tiles read cells that others update, so the step goes from one state plane set to the
// other (the host swaps them); once the run has ended a step copies the state.
// Measured per step with its control launch: 48^2 26 -> 15 us, 256^2 29 -> 18.6, 512^2 51 -> 37, 1024^2 134 -> 105,
// 2048 x 1500 392 -> 280.
#include "fvg_kernels_impl.hpp"

namespace fvg {

namespace {

constexpr int TX = kHancockTile, TY = kHancockTile;   // cells of a tile
constexpr int SX = TX + 2, SY = TY + 2;               // cells with advanced states
constexpr int WX = TX + 4, WY = TY + 4;               // cells with primitives
static_assert(SX * SY == 256 && (TX + 1) * TY <= 256 && WX * WY <= 512, "thread assignments of k_hancock_step2d");

struct Tile {
    double W[4][WY][WX];
    double S[4][4][SY][SX];          // advanced states: low x, high x, low y, high y side of the cell
    double Fx[4][TY][TX + 1], Fy[4][TY + 1][TX];
    int wide[8], wide_states[8];
};

// coordinate g (from -2) of a periodic axis of n cells; n may be smaller than the tile
__device__ __forceinline__ int wrapped(int g, int n) {
    g = g < 0 ? g + n : g;
    return g < n ? g : g % n;
}

// the advanced states of the cell at (lx, ly) of the S arrays; returns how many were inadmissible and kept; wide is set
// when an advanced one is not state_moderate
template <bool IR>
__device__ __forceinline__ int advance_states(const KP& p, Tile& s, int lx, int ly, double half_dt, bool& wide) {
    constexpr int NV = 4;
    double st[4][NV];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        double lo[NV], hi[NV];
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const double wm = d == 0 ? s.W[q][ly + 1][lx] : s.W[q][ly][lx + 1], w0 = s.W[q][ly + 1][lx + 1],
                         wp = d == 0 ? s.W[q][ly + 1][lx + 2] : s.W[q][ly + 2][lx + 1];
            lo[q] = muscl_wr<IR>(p.lim, wm, w0, wp);
            hi[q] = muscl_wl<IR>(p.lim, wm, w0, wp);
        }
        p2c<NV, IR>(p.rs.eos, lo, st[2 * d]);
        p2c<NV, IR>(p.rs.eos, hi, st[2 * d + 1]);
    }
    const double hx = half_dt / p.dx, hy = half_dt / p.dy;
    double f[4][NV], dd[NV];
#pragma unroll
    for (int k = 0; k < 4; ++k) euler_flux_axis<NV, IR>(p.rs.eos, st[k], k / 2, f[k]);
#pragma unroll
    for (int q = 0; q < NV; ++q) dd[q] = hx * (f[1][q] - f[0][q]) + hy * (f[3][q] - f[2][q]);
    int kept = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        double nw[NV];
#pragma unroll
        for (int q = 0; q < NV; ++q) nw[q] = st[k][q] - dd[q];
        const bool ok = admissible<NV>(p, nw);
        kept += ok ? 0 : 1;
        wide |= ok & !state_moderate(nw);
#pragma unroll
        for (int q = 0; q < NV; ++q) s.S[k][q][ly][lx] = ok ? nw[q] : st[k][q];
    }
    return kept;
}

// the flux of one face of the tile; returns its wave speed
template <int D, bool IR>
__device__ __forceinline__ double tile_face(const KP& p, Tile& s, int fi, int fj) {
    double UL[4], UR[4], F[4], sm;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        UL[q] = D == 0 ? s.S[1][q][fj + 1][fi] : s.S[3][q][fj][fi + 1];
        UR[q] = D == 0 ? s.S[0][q][fj + 1][fi + 1] : s.S[2][q][fj + 1][fi + 1];
    }
    face_flux<4, IR>(p.rs, UL, UR, D, F, sm);
#pragma unroll
    for (int q = 0; q < 4; ++q) (D == 0 ? s.Fx[q][fj][fi] : s.Fy[q][fj][fi]) = F[q];
    return sm;
}

}   // namespace

__global__ __launch_bounds__(512) void k_hancock_step2d(KP p, const double* __restrict__ U0, double* __restrict__ out) {
    __shared__ Tile s;
    const int t = threadIdx.x, i0 = blockIdx.x * TX, j0 = blockIdx.y * TY;
    // the thread's cell of the primitives and, of the first TX * TY threads, its cell of the tile
    const int wi = t % WX, wj = t / WX;
    double u[4], own[4];
    if (t < WX * WY) {
        const long long c = (long long)wrapped(j0 - 2 + wj, p.ny) * p.nx + wrapped(i0 - 2 + wi, p.nx);
#pragma unroll
        for (int q = 0; q < 4; ++q) u[q] = U0[q * p.nc + c];
    }
    const int ci = i0 + t % TX, cj = j0 + t / TX;
    const bool mine = t < TX * TY && ci < p.nx && cj < p.ny;
    const long long c = (long long)cj * p.nx + ci;
    if (mine)
#pragma unroll
        for (int q = 0; q < 4; ++q) own[q] = U0[q * p.nc + c];
    if (p.st->done) {   // uniform: the run has ended, the state moves on as it is
        if (mine)
#pragma unroll
            for (int q = 0; q < 4; ++q) out[q * p.nc + c] = own[q];
        return;
    }
    const double half_dt = p.st->half_dt, dt = p.st->dt;
    bool wide = false;
    if (t < WX * WY) {
        double w[4];
        c2p<4>(p.rs.eos, u, w, (double*)nullptr);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            s.W[q][wj][wi] = w[q];
            wide |= !value_in_range(w[q]);
        }
    }
    const bool any = __any(wide);
    if ((t & 63) == 0) s.wide[t >> 6] = any;
    __syncthreads();
    int nwide = 0;   // every value this tile reads is in range, or none of the in-range operations is used
#pragma unroll
    for (int k = 0; k < 8; ++k) nwide |= s.wide[k];
    bool ir = p.ir != 0 && __builtin_amdgcn_readfirstlane(nwide) == 0;
    wide = false;
    if (t < SX * SY) {
        const int lx = t % SX, ly = t / SX;
        const int kept = ir ? advance_states<true>(p, s, lx, ly, half_dt, wide) : advance_states<false>(p, s, lx, ly, half_dt, wide);
        const int gi = i0 + lx - 1, gj = j0 + ly - 1;
        if (kept && lx >= 1 && lx <= TX && ly >= 1 && ly <= TY && gi < p.nx && gj < p.ny)
            atomicAdd((unsigned long long*)&p.st->reverted, (unsigned long long)kept);
    }
    const bool any_state = __any(wide);
    if ((t & 63) == 0) s.wide_states[t >> 6] = any_state;
    __syncthreads();
    nwide = 0;
#pragma unroll
    for (int k = 0; k < SX * SY / 64; ++k) nwide |= s.wide_states[k];
    ir = ir && __builtin_amdgcn_readfirstlane(nwide) == 0;
    double speed = 0.0;   // a face beyond the mesh in a ragged tile is a face of the wrapped cells
    const int h = t & 255;
    if (t < 256) {
        if (h < (TX + 1) * TY) {
            const int fi = h % (TX + 1), fj = h / (TX + 1);
            speed = ir ? tile_face<0, true>(p, s, fi, fj) : tile_face<0, false>(p, s, fi, fj);
        }
    } else if (h < TX * (TY + 1)) {
        const int fi = h % TX, fj = h / TX;
        speed = ir ? tile_face<1, true>(p, s, fi, fj) : tile_face<1, false>(p, s, fi, fj);
    }
    double local = 0.0;
    if (speed > local) local = speed;
    __syncthreads();
    if (mine) {
        const int x = t % TX, y = t / TX;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double fl = s.Fx[q][y][x], fr = s.Fx[q][y][x + 1], fb = s.Fy[q][y][x], ft = s.Fy[q][y + 1][x];
            const double R = ((0.0 - (fr * p.Ax - fl * p.Ax)) - (ft * p.Ay - fb * p.Ay)) * p.inv_vol;
            out[q * p.nc + c] = own[q] + dt * R;
        }
    }
    block_max_to(local, p.spd + ((size_t)SPD_CONV * kSpeedSlots + (blockIdx.y * gridDim.x + blockIdx.x) % kSpeedSlots) * kSlotStride);
}

}   // namespace fvg
