// k_adjoint.hip — reverse-time adjoint of one FP64 explicit-Euler step of the
// snowflake and sintering models.
//
// Given the state u before a step, the state u' after it and the cotangent
// lam' = dJ/du', the kernels produce lam = dJ/du (the transposed Jacobian of
// the step applied to lam') and add the step's contribution to dJ/dp for the
// differentiable parameters.  They transpose exactly the arithmetic of the
// forward sweeps (same stencils, same anisotropy evaluation, same noise):
// every forward read of a neighbour through the boundary map bmap becomes, in
// the adjoint, a gather over the pre-images {j : bmap(j + d) = i}, so zero-flux
// mirrors and periodic wrap transpose without special cases.
//
// A step is one kernel with one workgroup per tile: the intermediate
// cotangents live in LDS, evaluated on the tile and the ring of cells around
// it that the next stage reads (the rings overlap between tiles; their cells
// are evaluated again by each).  Parameter partial sums are reduced per
// workgroup and added to a per-tile accumulator slot, so the sums are
// deterministic.
//
// Snowflake (forward: snowflake/function.h:5-60 restated in k_snowflake.hip):
//   mu      = dt/tau (lam_phi' + K lam_T')                   cotangent of the bracket
//   lamP_e  = 1/(2dy) (sum mu over rows whose +y read is e  - ... -y read is e)
//   lamQ_e  = -1/(2dx) (same along x)
//   lamE2_e = mu_e lap(phi)_e
//   -> lam(eps), lam(eps'), lam(theta) -> lam(gx), lam(gy) at every cell
//   lam_phi = lam_phi' + mu (dR/dphi + dN/dphi) + div^T(lam g) + lap^T(E2 mu)
//   lam_T   = lam_T'  + mu phi(1-phi) dm/dT + dt lap^T(lam_T')
// Sintering (forward: sintering/function.h:51-159, order of main.cu:136-146):
//   the clamps pass the cotangent where 0 <= v < 1 and stop it elsewhere;
//   the eta updates read the NEW c, so their cotangent flows into c' first.
#include "kernels.hpp"
#include "tile_common.hpp"
#include "sf_math.hpp"

namespace amps {

// Calls f(j) for every j in [0, n) with bmap(j + d, n, bc) == i.
template <class F>
__device__ inline void for_preimages(int i, int d, int n, int bc, F&& f) {
    if (bc == AMPS_BC_PERIODIC) {
        int j = i - d;
        if (j < 0) j += n;
        else if (j >= n) j -= n;
        f(j);
        return;
    }
    int j = i - d;
    if (j >= 0 && j < n) f(j);
    if (i > 0) {  // left mirror: j + d < 0, -(j + d) == i
        j = -i - d;
        if (j >= 0 && j < n && j + d < 0) f(j);
    }
    if (i < n - 1) {  // right mirror: j + d >= n, 2(n-1) - (j + d) == i
        j = 2 * (n - 1) - i - d;
        if (j >= 0 && j < n && j + d >= n) f(j);
    }
}

// Box of a TS x TS tile with an H-cell halo in LDS, addressed by tile
// coordinates (y, x) in [-H, TS + H); frame(r): halo cell r of the NF.
template <int TS, int H>
struct AdjBox {
    static constexpr int LW = TS + 2 * H, SZ = LW * LW, NF = SZ - TS * TS;
    __device__ static inline int at(int y, int x) { return (y + H) * LW + x + H; }
    __device__ static inline void frame(int r, int& y, int& x) {
        if (r < 2 * H * LW) {
            const int row = r / LW;
            x = r - row * LW - H;
            y = (row < H ? row : TS + row) - H;
        } else {
            const int q = r - 2 * H * LW, j = q % (2 * H);
            y = q / (2 * H);
            x = j < H ? j - H : TS + j - H;
        }
    }
};

// Cell (gy, gx) of instance D, boundary-mapped.
__device__ inline int adj_cell(const InstDesc& D, int gy, int gx) {
    const bool per = D.bc == AMPS_BC_PERIODIC;
    return map_cell(gy, D.ny, per) * D.nx + map_cell(gx, D.nx, per);
}

// Tile origin of the transposed reads.  MIRROR: the tile meets a zero-flux
// edge and its reads walk the pre-images; elsewhere the pre-image of a read
// at distance d is the cell at distance -d of the box (the halo of a
// periodic grid holds the wrapped values).
struct AdjEdge {
    int oy, ox, ny, nx;
};
__device__ inline bool adj_mirror(const InstDesc& D, int oy, int ox, int ts) {
    return D.bc != AMPS_BC_PERIODIC && (oy == 0 || ox == 0 || oy + ts == D.ny || ox + ts == D.nx);
}

// Sum over the pre-images along x (row y fixed) and along y of a read at
// distance d, and the transposed Laplacian without its 1/(dx dy) factor: the
// pre-image values of the stencil's offsets minus centre weight times b(y, x).
// A ring cell outside a zero-flux domain has no meaning and no reader: its
// gather only has to stay inside the box.
template <int TS, int H, bool MIRROR>
__device__ inline double adj_gather_x(const double* b, int y, int x, int d, const AdjEdge& ed) {
    if constexpr (!MIRROR) return b[AdjBox<TS, H>::at(y, x - d)];
    double s = 0.0;
    for_preimages(ed.ox + x, d, ed.nx, AMPS_BC_NEUMANN, [&](int j) {
        const int r = j - ed.ox;
        if (r >= -H && r < TS + H) s += b[AdjBox<TS, H>::at(y, r)];
    });
    return s;
}
template <int TS, int H, bool MIRROR>
__device__ inline double adj_gather_y(const double* b, int y, int x, int d, const AdjEdge& ed) {
    if constexpr (!MIRROR) return b[AdjBox<TS, H>::at(y - d, x)];
    double s = 0.0;
    for_preimages(ed.oy + y, d, ed.ny, AMPS_BC_NEUMANN, [&](int j) {
        const int r = j - ed.oy;
        if (r >= -H && r < TS + H) s += b[AdjBox<TS, H>::at(r, x)];
    });
    return s;
}
template <int TS, int H, bool MIRROR>
__device__ inline double adj_lapT(const double* b, int y, int x, bool ref, const AdjEdge& ed) {
    double s = adj_gather_x<TS, H, MIRROR>(b, y, x, -1, ed) + adj_gather_x<TS, H, MIRROR>(b, y, x, 1, ed) +
               adj_gather_y<TS, H, MIRROR>(b, y, x, -1, ed) + adj_gather_y<TS, H, MIRROR>(b, y, x, 1, ed);
    double w0 = 4.0;
    if constexpr (H >= 2) {
        if (ref) {
            s += adj_gather_x<TS, H, MIRROR>(b, y, x, -2, ed) + adj_gather_x<TS, H, MIRROR>(b, y, x, 2, ed) +
                 adj_gather_y<TS, H, MIRROR>(b, y, x, -2, ed) + adj_gather_y<TS, H, MIRROR>(b, y, x, 2, ed);
            w0 = 8.0;
        }
    }
    return s - w0 * b[AdjBox<TS, H>::at(y, x)];
}

// Workgroup sum of NG partials over NW waves; thread 0 adds them to
// acc[g][tile].
template <int NG, int NW = WG / 64>
__device__ inline void block_accumulate(double (&v)[NG], double* acc, int total_tiles, int tile, double* red) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        double x = v[g];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
        if ((threadIdx.x & 63) == 0) red[g * NW + (threadIdx.x >> 6)] = x;
    }
    __syncthreads();
    if (threadIdx.x < NG) {
        const int g = threadIdx.x;
        double s = red[g * NW];
#pragma unroll
        for (int i = 1; i < NW; ++i) s += red[g * NW + i];
        acc[(size_t)g * total_tiles + tile] += s;
    }
}

// ============================================================== snowflake
// gradient slots: 0 delta, 1 K, 2 epsb, 3 tau
constexpr int SF_NG = 4;

// Boxes of the fused reverse step in LDS for a Laplacian of reach S: phi
// halo 2S, mu and lam_T' S + 1, the cotangents of the gradient (w1, w2) and
// E2 mu (w3) S.  Tile 32: 67 KB at S = 2, 58.8 KB at S = 1 (two 512-thread
// workgroups per CU); tile 16: 22 KB at S = 2.
template <int TS, int NT, int S>
struct SfAdjLds {
    double phi[AdjBox<TS, 2 * S>::SZ];
    double mu[AdjBox<TS, S + 1>::SZ], lt[AdjBox<TS, S + 1>::SZ];
    double w1[AdjBox<TS, S>::SZ], w2[AdjBox<TS, S>::SZ], w3[AdjBox<TS, S>::SZ];
    double red[NT / 64 * SF_NG];
};

// w1 = lam(gx), w2 = lam(gy) and w3 = E2 mu at box cell (y, x) (halo S);
// OWN: the tile's partials of delta and epsb.
template <int TS, int NT, int S, bool MIRROR, bool OWN>
__device__ inline void sf_adj_grad(SfAdjLds<TS, NT, S>& L, const InstDesc& D, const AdjEdge& ed, int y, int x,
                                   bool ref, double (&g)[SF_NG]) {
    using P = AdjBox<TS, 2 * S>;
    const int n = (int)D.k[SFK_ANISO_N];
    const double inv2dx = D.k[SFK_INV_2DX], inv2dy = D.k[SFK_INV_2DY];
    const double cth0 = D.k[SFK_COS_N_THETA0], sth0 = D.k[SFK_SIN_N_THETA0];
    const double epsb = D.k[SFK_EPSB], epsbd = D.k[SFK_EPSB_DELTA], mend = D.k[SFK_MEPSB_ANISO_DELTA];
    const double* f = L.phi + P::at(y, x);
    constexpr int LW = P::LW;
    const double gx = (f[1] - f[-1]) * inv2dx;
    const double gy = (f[LW] - f[-LW]) * inv2dy;
    double c, s;
    sf_unit_power<double>(gx, gy, n, c, s);
    const double ca = c * cth0 + s * sth0, sa = s * cth0 - c * sth0;
    const double eps = epsb + epsbd * ca, epsd = mend * sa;
    const double A = eps * epsd;
    const double lamP = inv2dy * (adj_gather_y<TS, S + 1, MIRROR>(L.mu, y, x, 1, ed) -
                                  adj_gather_y<TS, S + 1, MIRROR>(L.mu, y, x, -1, ed));
    const double lamQ = -inv2dx * (adj_gather_x<TS, S + 1, MIRROR>(L.mu, y, x, 1, ed) -
                                   adj_gather_x<TS, S + 1, MIRROR>(L.mu, y, x, -1, ed));
    const double mue = L.mu[AdjBox<TS, S + 1>::at(y, x)];
    double lap;
    if (S == 2 && ref)
        lap = (f[-1] + f[-2] + f[1] + f[2] + f[-LW] + f[-2 * LW] + f[LW] + f[2 * LW] - 8.0 * f[0]) *
              D.k[SFK_INV_DXDY];
    else
        lap = (f[-1] + f[1] + f[-LW] + f[LW] - 4.0 * f[0]) * D.k[SFK_INV_DXDY];
    const double lamE2 = mue * lap;
    const double lamA = lamP * gx + lamQ * gy;
    const double lame = 2.0 * eps * lamE2 + epsd * lamA;
    const double lamd = eps * lamA;
    const double lamth = lame * epsd + lamd * ((double)n * mend * ca);
    // d theta / d(gx, gy) = (-gy, gx) / |g|^2, evaluated on the rescaled
    // gradient; the cotangent is multiplied in before the power-of-two
    // scale 2^-e, which overflows on its own for subnormal gradients (a
    // zero cotangent then gives 0, not 0 * inf)
    double thx = 0.0, thy = 0.0;
    const double mx = fmax(fabs(gx), fabs(gy));
    if (mx != 0.0) {
        int e;
        frexp(mx, &e);
        const double u = ldexp(gx, -e), v = ldexp(gy, -e);
        const double ir2 = 1.0 / (u * u + v * v);
        thx = ldexp(lamth * (-v * ir2), -e);
        thy = ldexp(lamth * (u * ir2), -e);
    }
    const int o = AdjBox<TS, S>::at(y, x);
    L.w1[o] = A * lamP + thx;
    L.w2[o] = A * lamQ + thy;
    L.w3[o] = eps * eps * mue;
    if (OWN) {
        const double delta = D.p[AMPS_SF_DELTA];
        g[0] += lame * (epsb * ca) + lamd * (-epsb * (double)n * sa);
        g[2] += lame * (1.0 + delta * ca) + lamd * (-(double)n * delta * sa);
    }
}

// The stages after staging: the gradient's cotangents on the tile and S
// cells around it, then the tile's lam_phi and lam_T.
template <int TS, int NT, int S, bool MIRROR, int OWN = TS * TS / NT>
__device__ inline void sf_adj_out(SfAdjLds<TS, NT, S>& L, const AdjArgs& a, const InstDesc& D, const AdjEdge& ed,
                                  const int (&cell)[OWN], const double (&lp0)[OWN], const double (&tv)[OWN],
                                  double (&g)[SF_NG]) {
    using W = AdjBox<TS, S>;
    static_assert(W::NF <= NT, "one frame cell per thread");
    const int tid = threadIdx.x;
    const bool ref = D.stencil == AMPS_STENCIL_REF;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT;
        sf_adj_grad<TS, NT, S, MIRROR, true>(L, D, ed, e / TS, e % TS, ref, g);
    }
    if (tid < W::NF) {
        int y, x;
        W::frame(tid, y, x);
        sf_adj_grad<TS, NT, S, MIRROR, false>(L, D, ed, y, x, ref, g);
    }
    __syncthreads();
    const double inv2dx = D.k[SFK_INV_2DX], inv2dy = D.k[SFK_INV_2DY], inv = D.k[SFK_INV_DXDY];
    const double dt = D.k[SFK_DT], aop = D.k[SFK_ALPHA_OVER_PI], gam = D.k[SFK_GAMMA], teq = D.k[SFK_TEQ];
    const double noise = D.k[SFK_NOISE];
    const uint32_t key = noise_key(D.seed, (uint64_t)(*a.step_ctr + a.step_add));
    double* lam = a.lam + D.cell_base;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT, y = e / TS, x = e % TS;
        const double p = L.phi[AdjBox<TS, 2 * S>::at(y, x)], t = tv[i];
        const double m_u = L.mu[AdjBox<TS, S + 1>::at(y, x)];
        const double arg = gam * (teq - t);
        const double m = aop * atan(arg);
        const double pp = p * (1.0 - p);
        double dR = (1.0 - 2.0 * p) * (p - 0.5 + m) + pp;
        if (noise != 0.0) {
            const double u = (double)noise_u24(key, (uint32_t)cell[i]);
            dR += noise * (1.0 - 2.0 * p) * (u - 0.5);
        }
        double lp = lp0[i] + m_u * dR;
        lp += inv2dx * (adj_gather_x<TS, S, MIRROR>(L.w1, y, x, 1, ed) - adj_gather_x<TS, S, MIRROR>(L.w1, y, x, -1, ed));
        lp += inv2dy * (adj_gather_y<TS, S, MIRROR>(L.w2, y, x, 1, ed) - adj_gather_y<TS, S, MIRROR>(L.w2, y, x, -1, ed));
        lp += inv * adj_lapT<TS, S, MIRROR>(L.w3, y, x, ref, ed);
        const double dmdT = aop * (-gam) / (1.0 + arg * arg);
        const double lt = L.lt[AdjBox<TS, S + 1>::at(y, x)] + m_u * pp * dmdT +
                          dt * inv * adj_lapT<TS, S + 1, MIRROR>(L.lt, y, x, ref, ed);
        lam[cell[i]] = lp;
        lam[a.total_cells + cell[i]] = lt;
    }
}

// One reverse step: a workgroup stages phi and both cotangents of its tile
// with their halos, forms mu = dt/tau (lam_phi' + K lam_T') on the way in,
// and writes the tile's lam_phi and lam_T: 56 B of state traffic per cell
// where three kernels over full-grid work arrays moved about 130.  512^2,
// tile 16, reach 2: 11.1 us a step against 25.4 for the three kernels (3.5 us
// of it a launch's fixed cost; the tiles' chains of rcp, ldexp and atan
// otherwise).
template <int TS, int NT, int S>
__global__ __launch_bounds__(NT, 4) void sf_adj_kernel(AdjArgs a) {
    using P = AdjBox<TS, 2 * S>;
    using M = AdjBox<TS, S + 1>;
    constexpr int OWN = TS * TS / NT, FP = (P::NF + NT - 1) / NT;
    static_assert(M::NF <= NT, "one frame cell per thread");
    __shared__ SfAdjLds<TS, NT, S> L;
    const int w = xcd_remap(blockIdx.x, gridDim.x);
    const InstDesc& D = a.inst[a.tile_inst[w]];
    const int lti = w - D.tile_base, tyi = lti / D.tx;
    const int oy = tyi * TS, ox = (lti - tyi * D.tx) * TS;
    const size_t TC = a.total_cells;
    const double* u = a.u + D.cell_base;
    const double* un = a.un + D.cell_base;
    const double* ln = a.lam_n + D.cell_base;
    const int tid = threadIdx.x;
    const double dtt = D.k[SFK_DT_OVER_TAU], K = D.k[SFK_KAPPA], tau = D.p[AMPS_SF_TAU];
    // every load of the tile in flight before the first LDS store
    double pv[OWN], pn[OWN], tv[OWN], lp[OWN], lt[OWN], fp[FP], fl, ft;
    int cell[OWN], py[FP], px[FP], my, mx;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT;
        cell[i] = (oy + e / TS) * D.nx + ox + e % TS;
        lp[i] = ln[cell[i]];
        lt[i] = ln[TC + cell[i]];
        pv[i] = u[cell[i]];
        pn[i] = un[cell[i]];
        tv[i] = u[TC + cell[i]];
    }
#pragma unroll
    for (int k = 0; k < FP; ++k) {
        P::frame(tid + k * NT < P::NF ? tid + k * NT : 0, py[k], px[k]);
        fp[k] = u[adj_cell(D, oy + py[k], ox + px[k])];
    }
    M::frame(tid < M::NF ? tid : 0, my, mx);
    {
        const int c = adj_cell(D, oy + my, ox + mx);
        fl = ln[c];
        ft = ln[TC + c];
    }
    double g[SF_NG] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT, y = e / TS, x = e % TS;
        const double big = lp[i] + K * lt[i];
        L.phi[P::at(y, x)] = pv[i];
        L.mu[M::at(y, x)] = dtt * big;
        L.lt[M::at(y, x)] = lt[i];
        const double dphi = pn[i] - pv[i];
        g[1] += lt[i] * dphi;
        g[3] -= big * dphi / tau;
    }
#pragma unroll
    for (int k = 0; k < FP; ++k)
        if (tid + k * NT < P::NF) L.phi[P::at(py[k], px[k])] = fp[k];
    if (tid < M::NF) {
        const double big = fl + K * ft;
        L.mu[M::at(my, mx)] = dtt * big;
        L.lt[M::at(my, mx)] = ft;
    }
    __syncthreads();
    const AdjEdge ed{oy, ox, D.ny, D.nx};
    if (adj_mirror(D, oy, ox, TS)) sf_adj_out<TS, NT, S, true>(L, a, D, ed, cell, lp, tv, g);
    else sf_adj_out<TS, NT, S, false>(L, a, D, ed, cell, lp, tv, g);
    block_accumulate<SF_NG, NT / 64>(g, a.gacc, a.total_tiles, w, L.red);
}

// ============================================================== sintering
// gradient slots: 0 Dsurf, 1 Dgb, 2 kappa_c, 3 kappa_eta, 4 L, 5 Dvol
constexpr int SN_NG = 6;

// Boxes of the fused reverse step in LDS, by halo: c 4, etas and mu 3, Y 2,
// nu 1; lam_mu (halo 1) takes mu's place once every mu_lap is formed.  At
// tile 32: 76.8 KB, two 512-thread workgroups per CU.
template <int TS, int NT>
struct SnAdjLds {
    using C = AdjBox<TS, 4>;
    using E = AdjBox<TS, 3>;
    using Y2 = AdjBox<TS, 2>;
    using N1 = AdjBox<TS, 1>;
    double c[C::SZ];
    double e[2][E::SZ];
    double mu[E::SZ];
    double Y[Y2::SZ];
    double nu[2][N1::SZ];
    double red[NT / 64 * SN_NG];
};

// What a tile cell keeps from the mu_lap stage for the last one.
struct SnAdjOwn {
    double mu_lap, cn, kap;
};

// mu at box cell (y, x) (sintering/function.h:67-72).
template <int TS, int NT>
__device__ inline double sn_adj_mu(const SnAdjLds<TS, NT>& L, const InstDesc& D, int y, int x) {
    using C = AdjBox<TS, 4>;
    using E = AdjBox<TS, 3>;
    const int i = C::at(y, x), k = E::at(y, x);
    const double cv = L.c[i], a1 = L.e[0][k], a2 = L.e[1][k];
    const double con_lap =
        (L.c[i - 1] + L.c[i + 1] + L.c[i - C::LW] + L.c[i + C::LW] - 4.0 * cv) * D.k[SNK_INV_DXDY];
    const double sum2 = a1 * a1 + a2 * a2, sum3 = a1 * a1 * a1 + a2 * a2 * a2, om = 1.0 - cv;
    const double B = D.k[SNK_B], A2 = D.k[SNK_A2];
    const double df = B * (2.0 * cv + 4.0 * sum3 - 6.0 * sum2) - A2 * (cv * cv) * om + A2 * cv * (om * om);
    return df - D.k[SNK_HALF_KC] * con_lap;
}

// The stage of the clamp masks at box cell (y, x) (halo 2): Y = kappa dt M
// with kappa the cotangent of c's pre-clamp update, and nu_k of the etas'
// (halo 1).  ln: the three cotangents of the state after the step there.
// OWN: a tile cell, whose parameter partials are added to g and whose
// mu_lap, c' and kappa are kept.
template <int TS, int NT, bool OWN>
__device__ inline void sn_adj_mask(SnAdjLds<TS, NT>& L, const InstDesc& D, int y, int x, const double (&ln)[3],
                                   double (&g)[SN_NG], SnAdjOwn& own) {
    using E = AdjBox<TS, 3>;
    const int i = E::at(y, x);
    const double cv = L.c[AdjBox<TS, 4>::at(y, x)], a1 = L.e[0][i], a2 = L.e[1][i];
    const double inv = D.k[SNK_INV_DXDY], dt = D.k[SNK_DT], B = D.k[SNK_B];
    const double dtl = D.k[SNK_DT_L], hke = D.k[SNK_HALF_KE];
    const double mu_lap = (L.mu[i - 1] + L.mu[i + 1] + L.mu[i - E::LW] + L.mu[i + E::LW] - 4.0 * L.mu[i]) * inv;
    const double h = cv * cv * cv * (10.0 - 15.0 * cv + 6.0 * (cv * cv));
    const double mob = D.k[SNK_DVOL] * h + D.k[SNK_DVAP] * (1.0 - h) + D.k[SNK_DSURF] * cv * (1.0 - cv) +
                       D.k[SNK_DGB] * (a1 * a2 * 2.0);
    const double v = cv + dt * mob * mu_lap;
    const double cn = v >= 1.0 ? 1.0 : (v < 0.0 ? 0.0 : v);
    const double gc = (v >= 0.0 && v < 1.0) ? 1.0 : 0.0;
    const double sum2 = a1 * a1 + a2 * a2;
    double lcn = ln[0];
    const bool ring1 = OWN || (y >= -1 && y <= TS && x >= -1 && x <= TS);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const double ak = k == 0 ? a1 : a2;
        const double* e = L.e[k];
        const double l = (e[i - 1] + e[i + 1] + e[i - E::LW] + e[i + E::LW] - 4.0 * ak) * inv;
        const double dk = B * (-12.0 * (ak * ak) * (2.0 - cn) + 12.0 * ak * (1.0 - cn) + 12.0 * ak * sum2);
        const double wk = ak - dtl * (dk - hke * l);
        const double gk = (wk >= 0.0 && wk < 1.0) ? 1.0 : 0.0;
        const double nu = ln[1 + k] * gk;
        lcn += nu * (-dtl) * B * (12.0 * ak * ak - 12.0 * ak);
        if (ring1) L.nu[k][AdjBox<TS, 1>::at(y, x)] = nu;
        if (OWN) {
            g[3] += nu * dtl * 0.5 * l;             // d w_k / d kappa_eta
            g[4] += nu * (-dt) * (dk - hke * l);    // d w_k / d L
        }
    }
    const double kap = lcn * gc;
    L.Y[AdjBox<TS, 2>::at(y, x)] = kap * dt * mob;
    if (OWN) {
        own.mu_lap = mu_lap;
        own.cn = cn;
        own.kap = kap;
        const double q = kap * dt * mu_lap;
        g[0] += q * cv * (1.0 - cv);
        g[1] += q * (a1 * a2 * 2.0);
        g[5] += q * h;
    }
}

// The last two stages: lam_mu = lap^T(Y) on the tile and its ring, in mu's
// place, then the tile's cotangents; adds the kappa_c partial to g2.
template <int TS, int NT, bool MIRROR, int OWN = TS * TS / NT>
__device__ inline void sn_adj_out(SnAdjLds<TS, NT>& L, const InstDesc& D, const AdjEdge& ed,
                                  const SnAdjOwn (&own)[OWN], const int (&cell)[OWN], double& g2, double* lam,
                                  size_t TC) {
    using C = AdjBox<TS, 4>;
    using E = AdjBox<TS, 3>;
    using N1 = AdjBox<TS, 1>;
    const int tid = threadIdx.x;
    const double inv = D.k[SNK_INV_DXDY], dt = D.k[SNK_DT];
    double* lmu = L.mu;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT, y = e / TS, x = e % TS;
        const double lm = inv * adj_lapT<TS, 2, MIRROR>(L.Y, y, x, false, ed);
        lmu[N1::at(y, x)] = lm;
        const int k = C::at(y, x);
        const double l = (L.c[k - 1] + L.c[k + 1] + L.c[k - C::LW] + L.c[k + C::LW] - 4.0 * L.c[k]) * inv;
        g2 += lm * (-0.5) * l;
    }
    if (tid < N1::NF) {
        int y, x;
        N1::frame(tid, y, x);
        lmu[N1::at(y, x)] = inv * adj_lapT<TS, 2, MIRROR>(L.Y, y, x, false, ed);
    }
    __syncthreads();
    const double B = D.k[SNK_B], A2 = D.k[SNK_A2];
    const double dtl = D.k[SNK_DT_L], hke = D.k[SNK_HALF_KE], hkc = D.k[SNK_HALF_KC];
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT, y = e / TS, x = e % TS;
        const int k = E::at(y, x), r = N1::at(y, x);
        const double cv = L.c[C::at(y, x)], a1 = L.e[0][k], a2 = L.e[1][k], om = 1.0 - cv;
        const double cn = own[i].cn, kap = own[i].kap, lm = lmu[r];
        const double hp = 3.0 * cv * cv * (10.0 - 15.0 * cv + 6.0 * (cv * cv)) + cv * cv * cv * (-15.0 + 12.0 * cv);
        const double dMdc = (D.k[SNK_DVOL] - D.k[SNK_DVAP]) * hp + D.k[SNK_DSURF] * (1.0 - 2.0 * cv);
        const double dfdc = 2.0 * B - A2 * (2.0 * cv * om - cv * cv) + A2 * (om * om - 2.0 * cv * om);
        const double q = kap * dt * own[i].mu_lap;
        lam[cell[i]] = kap + q * dMdc + lm * dfdc - hkc * inv * adj_lapT<TS, 1, MIRROR>(lmu, y, x, false, ed);
        const double sum2 = a1 * a1 + a2 * a2;
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const double ak = f == 0 ? a1 : a2, aj = f == 0 ? a2 : a1;
            const double nuk = L.nu[f][r], nuj = L.nu[1 - f][r];
            const double ddk = B * (-24.0 * ak * (2.0 - cn) + 12.0 * (1.0 - cn) + 12.0 * sum2 + 24.0 * ak * ak);
            double la = nuk * (1.0 - dtl * ddk) + nuj * (-dtl) * B * 24.0 * aj * ak;
            la += q * D.k[SNK_DGB] * 2.0 * aj + lm * B * (12.0 * ak * ak - 12.0 * ak);
            la += dtl * hke * inv * adj_lapT<TS, 1, MIRROR>(L.nu[f], y, x, false, ed);
            lam[(size_t)(1 + f) * TC + cell[i]] = la;
        }
    }
}

// One reverse step: a workgroup stages c (halo 4), the etas (3) and the
// cotangents (2), evaluates mu on the tile and 3 cells around it, Y on 2, nu
// and lam_mu on 1, and writes the tile's three cotangents: 72 B of state
// traffic per cell where four kernels over full-grid work arrays moved about
// 250.  The re-evaluated rings cost 1.41x (mu), 1.27x (masks) and 1.13x
// (lam_mu) of a tile's arithmetic at tile 32.  1024^2: 32 us a step against
// 78 for the four kernels; bound by the latency of its five stages at 16
// waves per CU (LDS and 126 VGPRs), about 14 us of VALU issue.  Tile 16 (5
// waves per SIMD, rings 1.89x/1.56x/1.27x): 37 us.
template <int TS, int NT>
__global__ __launch_bounds__(NT, 4) void sn_adj_kernel(AdjArgs a) {
    using C = AdjBox<TS, 4>;
    using E = AdjBox<TS, 3>;
    using Y2 = AdjBox<TS, 2>;
    constexpr int OWN = TS * TS / NT, FC = (C::NF + NT - 1) / NT;
    static_assert(E::NF <= NT, "one frame cell per thread");
    __shared__ SnAdjLds<TS, NT> L;
    const int w = xcd_remap(blockIdx.x, gridDim.x);
    const InstDesc& D = a.inst[a.tile_inst[w]];
    const int lt = w - D.tile_base, tyi = lt / D.tx;
    const int oy = tyi * TS, ox = (lt - tyi * D.tx) * TS;
    const size_t TC = a.total_cells;
    const double* u = a.u + D.cell_base;
    const double* ln = a.lam_n + D.cell_base;
    const int tid = threadIdx.x;
    // the boxes' loads in flight together before the first LDS store
    double vc[OWN], ve[2][OWN], vl[OWN][3], fc[FC], fe[2], fl[3];
    int cell[OWN];
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT;
        cell[i] = (oy + e / TS) * D.nx + ox + e % TS;
        vc[i] = u[cell[i]];
        ve[0][i] = u[TC + cell[i]];
        ve[1][i] = u[2 * TC + cell[i]];
    }
    int cy[FC], cx[FC], ey, ex, yy, yx;
#pragma unroll
    for (int k = 0; k < FC; ++k) {
        C::frame(tid + k * NT < C::NF ? tid + k * NT : 0, cy[k], cx[k]);
        fc[k] = u[adj_cell(D, oy + cy[k], ox + cx[k])];
    }
    {
        E::frame(tid < E::NF ? tid : 0, ey, ex);
        const int g = adj_cell(D, oy + ey, ox + ex);
        fe[0] = u[TC + g];
        fe[1] = u[2 * TC + g];
    }
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT, y = e / TS, x = e % TS;
        L.c[C::at(y, x)] = vc[i];
        L.e[0][E::at(y, x)] = ve[0][i];
        L.e[1][E::at(y, x)] = ve[1][i];
    }
#pragma unroll
    for (int k = 0; k < FC; ++k)
        if (tid + k * NT < C::NF) L.c[C::at(cy[k], cx[k])] = fc[k];
    if (tid < E::NF) {
        L.e[0][E::at(ey, ex)] = fe[0];
        L.e[1][E::at(ey, ex)] = fe[1];
    }
    // the cotangents arrive during the mu stage
#pragma unroll
    for (int i = 0; i < OWN; ++i)
#pragma unroll
        for (int f = 0; f < 3; ++f) vl[i][f] = ln[f * TC + cell[i]];
    {
        Y2::frame(tid < Y2::NF ? tid : 0, yy, yx);
        const int g = adj_cell(D, oy + yy, ox + yx);
#pragma unroll
        for (int f = 0; f < 3; ++f) fl[f] = ln[f * TC + g];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT, y = e / TS, x = e % TS;
        L.mu[E::at(y, x)] = sn_adj_mu<TS, NT>(L, D, y, x);
    }
    if (tid < E::NF) L.mu[E::at(ey, ex)] = sn_adj_mu<TS, NT>(L, D, ey, ex);
    __syncthreads();
    double g[SN_NG] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    SnAdjOwn own[OWN];
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int e = tid + i * NT;
        sn_adj_mask<TS, NT, true>(L, D, e / TS, e % TS, vl[i], g, own[i]);
    }
    if (tid < Y2::NF) {
        SnAdjOwn unused;
        sn_adj_mask<TS, NT, false>(L, D, yy, yx, fl, g, unused);
    }
    __syncthreads();
    const AdjEdge ed{oy, ox, D.ny, D.nx};
    double* lam = a.lam + D.cell_base;
    if (adj_mirror(D, oy, ox, TS)) sn_adj_out<TS, NT, true>(L, D, ed, own, cell, g[2], lam, TC);
    else sn_adj_out<TS, NT, false>(L, D, ed, own, cell, g[2], lam, TC);
    block_accumulate<SN_NG, NT / 64>(g, a.gacc, a.total_tiles, w, L.red);
}

// ------------------------------------------------------------ host launch
int launch_adjoint_step(const AdjArgs& a, int model, int tile, hipStream_t s) {
    const dim3 g(a.total_tiles);
    if (tile != 16 && tile != 32) return AMPS_E_UNSUPPORTED;
    if (model == AMPS_SNOWFLAKE) {
        // S: the reach of the widest Laplacian among the instances
        if (tile == 16) {
            if (a.t_halo == 2) hipLaunchKernelGGL((sf_adj_kernel<16, 256, 2>), g, dim3(256), 0, s, a);
            else hipLaunchKernelGGL((sf_adj_kernel<16, 256, 1>), g, dim3(256), 0, s, a);
        } else {
            if (a.t_halo == 2) hipLaunchKernelGGL((sf_adj_kernel<32, 512, 2>), g, dim3(512), 0, s, a);
            else hipLaunchKernelGGL((sf_adj_kernel<32, 512, 1>), g, dim3(512), 0, s, a);
        }
    } else if (model == AMPS_SINTERING) {
        if (tile == 16) hipLaunchKernelGGL((sn_adj_kernel<16, 256>), g, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((sn_adj_kernel<32, 512>), g, dim3(512), 0, s, a);
    } else {
        return AMPS_E_UNSUPPORTED;
    }
    return hipGetLastError() == hipSuccess ? AMPS_OK : AMPS_E_HIP;
}

}  // namespace amps
