// sifv_visc.hpp - face stresses of the explicit and semi-implicit solvers on
// the GPU: viscous stress (addViscousFluxes, src/ViscousFlux.cpp:25-303) and
// capillary stress (addSurfaceTensionFluxes, src/SurfaceTension.cpp:7-255),
// called from src/ExplicitSolver.cpp:523-535 and
// src/SemiImplicitSolver.cpp:509-520.
//
// visc_kernel writes, per interior cell, the stress part of the momentum and
// energy right-hand sides of the RK stage's state: the cell's 2*DIM faces in
// the reference's accumulation order (x low face -, x high face +, then y,
// then z), each face's stress row and work formed exactly as the reference
// forms them.  Both stresses use the same face stencil: normal derivatives
// from the two cells, transverse derivatives the mean of the two cells'
// central differences (transverse spacing of the high-side cell), so one set
// of cell loads serves both.
//   viscous:   tau = mu (grad u + grad u^T) - 2/3 mu div(u) I (face row),
//              mu scalar or the mean of the two cells' sum_k alpha_k mu_k;
//   capillary: from g = grad alpha_0, T_n = sigma (|g|^2 - g_n^2) / max(|g|, eps),
//              T_a = -sigma g_n g_a / max(|g|, eps);
//   work = (tau or T) . u_face, weighted by faceArea / cellVolume of the cell.
// The reference adds all viscous faces, then all capillary faces; here each
// face's two rows are summed first (a reassociation of the same terms).
// Velocities and volume fractions come from the stage's conservative buffer
// through the ghost mapping, as the stage kernels read them.  The stage update adds the
// result after the flux terms and the body force.
#pragma once

#include "sifv_stage.hpp"

namespace sifv {

template <typename T>
struct ViscArgs {
    StageParams<T> P;       // grid, EOS, mixture, source buffer P.src
    int viscous;            // hasViscosity
    double mu;              // scalar viscosity
    int nPhaseMu;           // > 0: face viscosity from alpha-weighted phase values
    double phaseMu[kMaxPhases];
    double sigma;           // > 0: capillary stress (multiphase states only)
    double capEps;          // epsGradAlpha
    double* out;            // DIM + 1 padded fields: momentum components, energy
};

// ---- Tiling -------------------------------------------------------------------
// A block owns 64 columns x kViscRows rows (256 columns in 1D) and marches
// kViscPlanes planes of z.  Each plane's velocities (and volume fraction and
// alpha-weighted viscosity of a multiphase state) are formed once per cell,
// one-cell halo included, and kept in LDS for the three planes k-1..k+1 a
// face stencil of plane k reaches; the high z face of a plane is the next
// plane's low one and stays in registers.
// What bounds it: loads and conservative-to-primitive divisions, so each cell
// is converted 1.6 times (xy halo and the two extra planes of a block) instead
// of once for each of the 60 stencil references its 6 faces make in 3D.
// 512 threads, 79 KB of LDS and at most 128 VGPRs (19 spilled) give the
// two-phase 3D form two blocks per CU; 8 planes per block leave a 160 x 144 x
// 176 mesh 1188 blocks.  Measured there (two-phase, both stresses): 1938 -> 268
// us per launch; 2D 501 x 333: 35 -> 10.7 us.  Small 3D meshes get few blocks (32^3:
// 16 on 256 CUs) and still gain: a two-phase step of 32^3 1259 -> 463 us.
constexpr int kViscCols = 64;
constexpr int kViscRows = 8;
constexpr int kViscPlanes = 8;
template <int DIM>
constexpr int visc_rows() { return DIM >= 2 ? kViscRows : 1; }
template <int DIM>
constexpr int visc_threads() { return DIM >= 2 ? kViscCols * kViscRows : 256; }

// Quotients by one positive denominator: its refined reciprocal and the
// residual-corrected quotient (div_fast with the reciprocal shared).
__device__ __forceinline__ double visc_quot(double a, double b, double r) {
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

// Per-cell values a face stencil reads.
template <int DIM, int NPH>
struct ViscCell {
    double u[DIM];
    double a0, mu;   // multiphase: alpha_0 and sum_k alpha_k mu_k
};

// Velocity (and alpha_0, mu) of the mapped cell; the velocity is the stage
// kernels' conversion (prim_of).  FP32 single-phase states convert in FP64 too.
template <int DIM, int NPH, typename T>
__device__ __forceinline__ void visc_load(const ViscArgs<T>& A, int i, int j, int k, ViscCell<DIM, NPH>& c) {
    const StageParams<T>& P = A.P;
    const Grid& g = P.g;
    bool fn[3] = {false, false, false}, ft[3] = {false, false, false};
    int si = i, sj = j, sk = k;
    const bool in = i >= 0 && i < g.nx && (DIM < 2 || (j >= 0 && j < g.ny)) && (DIM < 3 || (k >= 0 && k < g.nz));
    if (!in) {
        si = map_axis(clampi(i, -g.ngx, g.nx - 1 + g.ngx), g.nx, g.bc[0], g.bc[1], fn[0], ft[0]);
        if (DIM >= 2) sj = map_axis(clampi(j, -g.ngy, g.ny - 1 + g.ngy), g.ny, g.bc[2], g.bc[3], fn[1], ft[1]);
        if (DIM >= 3) sk = map_axis(clampi(k, -g.ngz, g.nz - 1 + g.ngz), g.nz, g.bc[4], g.bc[5], fn[2], ft[2]);
    }
    const size_t id = cell_index(g, si, sj, sk);
    auto ld = [&](int q) { return (double)P.src[(size_t)q * P.total + id]; };
    double rs;
    if constexpr (NPH == 0) {
        rs = ld(0);
    } else {
        rs = 0.0;
#pragma unroll
        for (int ph = 0; ph < NPH; ++ph) rs += ld(DIM + 2 + ph);
    }
    rs = dmax_ref(rs, 1e-14);
    const double ri = rcp_nr(rs);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        double u = visc_quot(ld(1 + d), rs, ri);
        bool f = fn[d];
#pragma unroll
        for (int e = 0; e < DIM; ++e)
            if (e != d) f = f != ft[e];
        c.u[d] = f ? -u : u;
    }
    if constexpr (NPH > 0) {
        c.a0 = ld(DIM + 2 + NPH);
        double m = 0.0;
        if (A.nPhaseMu > 0) {
#pragma unroll
            for (int ph = 0; ph < NPH; ++ph)
                if (ph < A.nPhaseMu) m += ld(DIM + 2 + NPH + ph) * A.phaseMu[ph];
        }
        c.mu = m;
    }
}

// Stress row and work of one face normal to DIR, added up: s[0..DIM-1] the
// momentum components, s[DIM] the work.  at(side, b, o) gives the stencil
// cell on the low (0) or high (1) side of the face, offset by o along the
// transverse axis b (o = 0: the cell itself).  rn = 1 / (normal distance of
// the two centroids), rt[b] = 1 / (2 h_b).
template <int DIM, int NPH, int DIR, typename T, typename F>
__device__ __forceinline__ void visc_face(const ViscArgs<T>& A, F&& at, double rn, const double* rt, double* s) {
    constexpr bool kCap = NPH > 0;
    const ViscCell<DIM, NPH> L = at(0, DIR, 0), R = at(1, DIR, 0);
    double grad[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    double ga[3] = {0, 0, 0};
#pragma unroll
    for (int a = 0; a < DIM; ++a) grad[a][DIR] = (R.u[a] - L.u[a]) * rn;
    if constexpr (kCap) ga[DIR] = (R.a0 - L.a0) * rn;
#pragma unroll
    for (int b = 0; b < DIM; ++b) {
        if (b == DIR) continue;
        const ViscCell<DIM, NPH> Lm = at(0, b, -1), Lp = at(0, b, 1), Rm = at(1, b, -1), Rp = at(1, b, 1);
#pragma unroll
        for (int a = 0; a < DIM; ++a) {
            if (!(a == b || a == DIR)) continue;
            grad[a][b] = 0.5 * ((Lp.u[a] - Lm.u[a]) * rt[b] + (Rp.u[a] - Rm.u[a]) * rt[b]);
        }
        if constexpr (kCap) ga[b] = 0.5 * ((Lp.a0 - Lm.a0) * rt[b] + (Rp.a0 - Rm.a0) * rt[b]);
    }
    double uf[3] = {0, 0, 0};
#pragma unroll
    for (int a = 0; a < DIM; ++a) uf[a] = 0.5 * (L.u[a] + R.u[a]);
    double st[3] = {0, 0, 0}, w = 0.0;
    if (A.viscous) {
        double divU = grad[0][0];
        if (DIM >= 2) divU += grad[1][1];
        if (DIM >= 3) divU += grad[2][2];
        double mu = A.mu;
        if constexpr (NPH > 0)
            if (A.nPhaseMu > 0) mu = 0.5 * (L.mu + R.mu);
#pragma unroll
        for (int a = 0; a < 3; ++a)
            st[a] = a == DIR ? mu * (2.0 * grad[DIR][DIR] - (2.0 / 3.0) * divU) : mu * (grad[a][DIR] + grad[DIR][a]);
        w = st[0] * uf[0] + st[1] * uf[1] + st[2] * uf[2];
    }
    if constexpr (kCap) {
        if (A.sigma > 0.0) {
            // |grad alpha| of a uniform region is 0: the square is kept in the
            // normal range (its root, 1e-145, is below every usable epsGradAlpha)
            const double q = dmax_ref(ga[0] * ga[0] + ga[1] * ga[1] + ga[2] * ga[2], 1e-290);
            const double ri = A.sigma * rcp_nr(dmax_ref(sqrt_fast(q), A.capEps));
            constexpr int b0 = DIR == 0 ? 1 : 0, b1 = DIR == 2 ? 1 : 2;
            double cap[3];
#pragma unroll
            for (int a = 0; a < 3; ++a)
                cap[a] = a == DIR ? (ga[b0] * ga[b0] + ga[b1] * ga[b1]) * ri : -(ga[DIR] * ga[a]) * ri;
            w += cap[0] * uf[0] + cap[1] * uf[1] + cap[2] * uf[2];
#pragma unroll
            for (int a = 0; a < 3; ++a) st[a] += cap[a];
        }
    }
#pragma unroll
    for (int a = 0; a < DIM; ++a) s[a] = st[a];
    s[DIM] = w;
}

template <int DIM, int NPH, typename T>
__global__ void __launch_bounds__(visc_threads<DIM>()) __attribute__((amdgpu_waves_per_eu(4, 8))) visc_kernel(ViscArgs<T> A) {
    const StageParams<T>& P = A.P;
    if (P.active && *P.active == 0) return;
    const Grid& g = P.g;
    constexpr int TX = DIM >= 2 ? kViscCols : 256, TY = visc_rows<DIM>();
    constexpr int HX = TX + 2, HY = DIM >= 2 ? TY + 2 : 1;
    constexpr int NF = DIM + (NPH > 0 ? 2 : 0);
    constexpr int NPL = DIM >= 3 ? 3 : 1;
    __shared__ double sv[NPL][NF][HY][HX];
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
    // blocks are dealt round-robin to the 8 XCDs: each takes a contiguous run
    const int nbx = (g.nx + TX - 1) / TX, nby = DIM >= 2 ? (g.ny + TY - 1) / TY : 1;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int bx = blk % nbx, by = (blk / nbx) % nby, bz = blk / (nbx * nby);
    const int i0 = bx * TX, j0 = by * TY;
    const int i = i0 + tx, j = j0 + ty;
    const int k0 = DIM >= 3 ? bz * kViscPlanes : 0, k1 = DIM >= 3 ? min(g.nz, k0 + kViscPlanes) : 1;
    const bool own = i < g.nx && j < g.ny;
    auto stage = [&](int k) {
        const int s = DIM >= 3 ? (k + 3) % 3 : 0;
        for (int m = tid; m < HX * HY; m += TX * TY) {
            const int a = m % HX, b = m / HX;
            const int ci = i0 - 1 + a, cj = DIM >= 2 ? j0 - 1 + b : 0;
            if (ci > g.nx || cj > g.ny) continue;   // past the last halo cell
            ViscCell<DIM, NPH> c;
            visc_load<DIM, NPH, T>(A, ci, cj, k, c);
#pragma unroll
            for (int d = 0; d < DIM; ++d) sv[s][d][b][a] = c.u[d];
            if constexpr (NPH > 0) {
                sv[s][DIM][b][a] = c.a0;
                sv[s][DIM + 1][b][a] = c.mu;
            }
        }
    };
    // stencil cell at (tx + di, ty + dj) of plane slot s
    auto get = [&](int s, int di, int dj) {
        ViscCell<DIM, NPH> c;
        const int a = tx + 1 + di, b = DIM >= 2 ? ty + 1 + dj : 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) c.u[d] = sv[s][d][b][a];
        if constexpr (NPH > 0) {
            c.a0 = sv[s][DIM][b][a];
            c.mu = sv[s][DIM + 1][b][a];
        }
        return c;
    };
    const int ic = own ? i : g.nx - 1, jc = own ? j : g.ny - 1;
    double h[3] = {g.dxw[ic + g.ngx], DIM >= 2 ? g.dyw[jc + g.ngy] : 1.0, 1.0};
    double rt[3] = {rcp_nr(2.0 * h[0]), rcp_nr(2.0 * h[1]), 0.5};
    const double rxl = rcp_nr(0.5 * (g.dxw[ic - 1 + g.ngx] + h[0])), rxh = rcp_nr(0.5 * (h[0] + g.dxw[ic + 1 + g.ngx]));
    double ryl = 0.0, ryh = 0.0;
    if constexpr (DIM >= 2) {
        ryl = rcp_nr(0.5 * (g.dyw[jc - 1 + g.ngy] + h[1]));
        ryh = rcp_nr(0.5 * (h[1] + g.dyw[jc + 1 + g.ngy]));
    }
    double zlo[DIM + 1];
    if constexpr (DIM >= 3) {
        stage(k0 - 1);
        stage(k0);
    } else {
        stage(0);
        __syncthreads();
    }
    for (int k = k0; k < k1; ++k) {
        if constexpr (DIM >= 3) {
            stage(k + 1);   // its slot held plane k-2
            __syncthreads();
            h[2] = g.dzw[k + g.ngz];
            rt[2] = rcp_nr(2.0 * h[2]);
        }
        if (own) {
            const int sc = DIM >= 3 ? k % 3 : 0, sm = DIM >= 3 ? (k + 2) % 3 : 0, sp = DIM >= 3 ? (k + 1) % 3 : 0;
            // faceArea / cellVolume with the reference's products
            const double rv = rcp_nr(h[0] * h[1] * h[2]);
            double acc[DIM + 1], s[DIM + 1];
#pragma unroll
            for (int q = 0; q <= DIM; ++q) acc[q] = 0.0;
            auto add = [&](double c) {
#pragma unroll
                for (int q = 0; q <= DIM; ++q) acc[q] += c * s[q];
            };
            // transverse offset (o along axis b) of a cell shifted by (x, y) in
            // plane slot `base` (slots sm, sc, sp along z)
            auto tr = [&](int x, int y, int z, int b, int o) {
                const int zz = z + (b == 2 ? o : 0);
                return get(zz < 0 ? sm : zz > 0 ? sp : sc, x + (b == 0 ? o : 0), y + (b == 1 ? o : 0));
            };
            const double cx = h[1] * h[2] * rv;
            visc_face<DIM, NPH, 0, T>(A, [&](int sd, int b, int o) { return tr(sd - 1, 0, 0, b, b == 0 ? 0 : o); }, rxl, rt, s);
            add(-cx);
            visc_face<DIM, NPH, 0, T>(A, [&](int sd, int b, int o) { return tr(sd, 0, 0, b, b == 0 ? 0 : o); }, rxh, rt, s);
            add(cx);
            if constexpr (DIM >= 2) {
                const double cy = h[0] * h[2] * rv;
                visc_face<DIM, NPH, 1, T>(A, [&](int sd, int b, int o) { return tr(0, sd - 1, 0, b, b == 1 ? 0 : o); }, ryl, rt, s);
                add(-cy);
                visc_face<DIM, NPH, 1, T>(A, [&](int sd, int b, int o) { return tr(0, sd, 0, b, b == 1 ? 0 : o); }, ryh, rt, s);
                add(cy);
            }
            if constexpr (DIM >= 3) {
                const double cz = h[0] * h[1] * rv;
                if (k == k0) {
                    const double rzl = rcp_nr(0.5 * (g.dzw[k - 1 + g.ngz] + h[2]));
                    visc_face<DIM, NPH, 2, T>(A, [&](int sd, int b, int o) { return tr(0, 0, sd - 1, b, b == 2 ? 0 : o); }, rzl, rt, zlo);
                }
#pragma unroll
                for (int q = 0; q <= DIM; ++q) s[q] = zlo[q];
                add(-cz);
                const double rzh = rcp_nr(0.5 * (h[2] + g.dzw[k + 1 + g.ngz]));
                visc_face<DIM, NPH, 2, T>(A, [&](int sd, int b, int o) { return tr(0, 0, sd, b, b == 2 ? 0 : o); }, rzh, rt, s);
                add(cz);
#pragma unroll
                for (int q = 0; q <= DIM; ++q) zlo[q] = s[q];
            }
            const size_t id = cell_index(g, i, j, k);
#pragma unroll
            for (int q = 0; q <= DIM; ++q) A.out[(size_t)q * P.total + id] = acc[q];
        }
        if constexpr (DIM >= 3) __syncthreads();   // plane k-1's slot is refilled next
    }
}

}  // namespace sifv
