// sifv_tile.hpp - the fused RK stage of a 2D mesh on workgroup tiles.
//
// Same work per cell as stage_xy_kernel (sifv_stage.hpp), split differently:
// a workgroup of NW waves owns 62 columns x (NW - 2) rows, one row per wave
// plus a halo row on either side (lane l <-> column X0-1+l, lanes 0 and 63 are
// halo columns).  Phases, separated by workgroup barriers:
//   1  every wave loads and converts its row; the two halo waves also the
//      R-1 rows beyond and the columns beyond the strip; primitives -> LDS;
//   2  each wave reconstructs its row's cells in y (plus state -> LDS) and,
//      if the row is owned, in x;
//   3  flux of the row's low y face (-> LDS) and of the x faces;
//   4  flux divergence, sources, stage update, dt of the new state.
// A wave of the marching kernel does two warm-up rows and then its rows one
// after the other, a serial chain of at least six rows' latency; here a row's
// chain is the whole kernel, which is what bounds meshes that leave the chip
// idle.  The price is two halo rows of y reconstruction per NW - 2 rows and
// the barriers.
#pragma once

#include "sifv_stage.hpp"

namespace sifv {

// Face-contribution slots the stage update of a full stage reads.
template <int DIM, int NPH, bool SEMI>
__device__ __forceinline__ constexpr bool face_slot_used(int q) {
    constexpr int NCV = DIM + 2 + 2 * NPH;
    if (q == NCV) return SEMI;                 // advected pressure
    if (q == NCV + 1) return SEMI || NPH > 0;  // divergence
    return part_slot_used<DIM, NPH, SEMI>(q);
}
template <int DIM, int NPH, bool SEMI>
constexpr int face_slots() {
    int n = 0;
    for (int q = 0; q < n_fc<DIM, NPH>(); ++q) n += face_slot_used<DIM, NPH, SEMI>(q) ? 1 : 0;
    return n;
}

template <int NPH, typename T>
constexpr int tile_min_waves() { return NPH > 0 ? 2 : 4; }

template <int R, int RS, int NPH, bool SEMI, typename T, bool SRC, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(tile_min_waves<NPH, T>(), 8)))
stage_tile_kernel(StageParams<T> P) {
    constexpr int DIM = 2;
    constexpr int NV = n_recon<DIM, NPH>();
    constexpr int NF = n_fc<DIM, NPH>();
    constexpr int NFU = face_slots<DIM, NPH, SEMI>();
    constexpr int NFL = DIM + 4 + NPH;
    constexpr int NCV = DIM + 2 + 2 * NPH;
    constexpr int E = R - 1;
    constexpr int TY = NW - 2;
    constexpr int ROWS = NW + 2 * E;    // prim rows: Y0-1-E .. Y0+TY+E
    constexpr int COLS = kWave + 2 * E;
    constexpr bool kSig = RS == RS_LF;
    constexpr int NS = NV + (kSig ? 1 : 0);

    if (P.active && *P.active == 0) return;
    const Grid& g = P.g;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int strip = blk / P.nseg;
    const int seg = blk - strip * P.nseg;
    const int X0 = strip * kOwn;
    const int col = X0 - 1 + lane;
    const int Y0 = seg * TY;
    const int r = Y0 - 1 + w;   // this wave's row
    const bool ownRow = w >= 1 && w <= TY && r < g.ny;
    const bool owned = ownRow && lane >= 1 && lane <= kOwn && col < g.nx;
    const bool useSig = kSig && P.igr;
    const bool incP = !SEMI;
    const bool igr = P.igr != 0;
    using C = CellT<T, NPH, SEMI>;

    // primitives of the tile; the y-face contributions take their place in phase 3
    constexpr int kPrim = NS * ROWS * COLS, kFace = NFU * (NW - 1) * kWave;
    __shared__ T buf[kPrim > kFace ? kPrim : kFace];
    __shared__ T plY[NS][NW - 1][kWave];           // plus states of rows Y0-1 .. Y0+TY-1
    __shared__ C up[NPH > 0 ? NPH + 1 : 1][NPH > 0 ? NW : 1][NPH > 0 ? kWave : 1];  // rho, alpha rho (upwinding)
    __shared__ double shMin[NW];
    auto prim = [&](int v, int row, int c) -> T& { return buf[(v * ROWS + row) * COLS + c]; };
    auto face = [&](int q, int row, int c) -> T& { return buf[(q * (NW - 1) + row) * kWave + c]; };

    const T eps = (T)P.eps;
    const int weno = P.weno;
    const double dt = *P.dt;
    const int cc = col < g.nx ? (col < 0 ? 0 : col) : g.nx - 1;
    const int rc = r < g.ny ? (r < 0 ? 0 : r) : g.ny - 1;
    const double dxc = g.dxw[cc + g.ngx], dyr = g.dyw[rc + g.ngy];

    // ---- phase 1 ----
    const bool xin = X0 - 1 - E >= 0 && X0 + kWave - 1 + E < g.nx;
    auto loadRaw = [&](int c, int row, RawCell<DIM, NPH, T>& q) __attribute__((always_inline)) {
        if (xin && row >= 0 && row < g.ny) {
            const size_t id = cell_index(g, c, row, 0);
#pragma unroll
            for (int f = 0; f < NCV; ++f) q.U[f] = P.src[(size_t)f * P.total + id];
            q.flip = 0;
        } else {
            load_raw<DIM, NPH, T>(P, P.src, c, row, 0, q);
        }
    };
    auto put = [&](const Cell<DIM, NPH, C>& c, int row, int pos, int ci, int cj) __attribute__((always_inline)) {
        T v[NV];
        recon_vars<DIM, NPH, T>(c, v);
#pragma unroll
        for (int q = 0; q < NV; ++q) prim(q, row, pos) = v[q];
        if constexpr (kSig)
            if (useSig) prim(NV, row, pos) = (T)load_sigma<DIM>(P, ci, cj, 0);
    };
    RawCell<DIM, NPH, T> raw;
    loadRaw(col, r, raw);
    T U0v[NCV];
    {
        const bool use0 = owned && P.c2 != 0.0;
        const size_t id = owned ? cell_index(g, col, r, 0) : 0;
#pragma unroll
        for (int q = 0; q < NCV; ++q) U0v[q] = use0 ? P.u0[(size_t)q * P.total + id] : T(0);
    }
    if (w == 0 || w == NW - 1) {
        // rows beyond the halo row, and the columns beyond the strip (those of
        // the lower half of the owned rows by wave 0, the others by the last wave)
        RawCell<DIM, NPH, T> ex[E > 0 ? E : 1];
#pragma unroll
        for (int e = 0; e < E; ++e) loadRaw(col, w == 0 ? r - 1 - e : r + 1 + e, ex[e]);
        RawCell<DIM, NPH, T> ec;
        constexpr int H0 = TY / 2;
        const int nrow = w == 0 ? H0 : TY - H0;
        const bool hasX = E > 0 && lane < 2 * E * nrow;
        const int hr = E > 0 ? lane / (2 * E > 0 ? 2 * E : 1) : 0, hq = lane - hr * 2 * E;
        const int hrow = (w == 0 ? 0 : H0) + hr;                               // owned row
        const int hcol = hq < E ? X0 - 1 - E + hq : X0 + kWave - 1 + (hq - E);
        if (hasX) loadRaw(hcol, Y0 + hrow, ec);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            Cell<DIM, NPH, C> c;
            raw_to_cell<DIM, NPH, T>(P, ex[e], c);
            put(c, w == 0 ? E - 1 - e : NW + E + e, lane + E, col, w == 0 ? r - 1 - e : r + 1 + e);
        }
        if (hasX) {
            Cell<DIM, NPH, C> c;
            raw_to_cell<DIM, NPH, T>(P, ec, c);
            put(c, 1 + E + hrow, hq < E ? hq : kWave + hq, hcol, Y0 + hrow);
        }
    }
    Cell<DIM, NPH, C> cur;
    raw_to_cell<DIM, NPH, T>(P, raw, cur);
    put(cur, w + E, lane + E, col, r);
    if constexpr (NPH > 0) {
        up[0][w][lane] = cur.rho;
#pragma unroll
        for (int ph = 0; ph < NPH; ++ph) up[1 + ph][w][lane] = cur.ar[ph];
    }
    __syncthreads();

    // ---- phase 2 ----
    T mY[NS], mX[NS], pX[NS];
    {
        T pl[NS];
        if constexpr (kSig) mY[NV] = pl[NV] = T(0);
        recon_set<R, T, NV>([&](int v, int s) __attribute__((always_inline)) { return prim(v, w + s, lane + E); }, eps,
                            weno, mY, pl);
        if (useSig)
            recon_set<R, T, 1>([&](int, int s) __attribute__((always_inline)) { return prim(NS - 1, w + s, lane + E); },
                               eps, weno, mY + NS - 1, pl + NS - 1);
        if (w < NW - 1) {
#pragma unroll
            for (int v = 0; v < NS; ++v) plY[v][w][lane] = pl[v];
        }
    }
    if (ownRow) {
        if constexpr (kSig) mX[NV] = pX[NV] = T(0);
        recon_set<R, T, NV>([&](int v, int s) __attribute__((always_inline)) { return prim(v, w + E, lane + s); }, eps,
                            weno, mX, pX);
        if (useSig)
            recon_set<R, T, 1>([&](int, int s) __attribute__((always_inline)) { return prim(NS - 1, w + E, lane + s); },
                               eps, weno, mX + NS - 1, pX + NS - 1);
    }
    __syncthreads();

    // ---- phase 3 ----
    T Glo[NF], FCx[NF], FCl[NF];
    if (w >= 1) {
        T pv[NS];
#pragma unroll
        for (int v = 0; v < NS; ++v) pv[v] = plY[v][w - 1][lane];
        FaceState<DIM, NPH, T> L, Rr;
        face_state<DIM, NPH, T>(P, pv, kSig ? pv[NS - 1] : T(0), L);
        face_state<DIM, NPH, T>(P, mY, kSig ? mY[NS - 1] : T(0), Rr);
        T F[NFL];
        riemann<RS, 1, DIM, NPH, T>(L, Rr, incP, igr, F);
        C rhoL = C(0), arL[NPH > 0 ? NPH : 1];
        if constexpr (NPH > 0) {
            rhoL = up[0][w - 1][lane];
#pragma unroll
            for (int ph = 0; ph < NPH; ++ph) arL[ph] = up[1 + ph][w - 1][lane];
        }
        face_contrib<DIM, NPH, T>(F, rhoL, cur.rho, arL, cur.ar, Glo);
        int n = 0;
#pragma unroll
        for (int q = 0; q < NF; ++q)
            if (face_slot_used<DIM, NPH, SEMI>(q)) face(n++, w - 1, lane) = Glo[q];
    }
    if (ownRow) {
        // face col+1/2: left = plus of this lane, right = minus of lane+1
        T nX[NS];
#pragma unroll
        for (int v = 0; v < NS; ++v) nX[v] = __shfl_down(mX[v], 1, kWave);
        FaceState<DIM, NPH, T> L, Rr;
        face_state<DIM, NPH, T>(P, pX, kSig ? pX[NS - 1] : T(0), L);
        face_state<DIM, NPH, T>(P, nX, kSig ? nX[NS - 1] : T(0), Rr);
        T F[NFL];
        riemann<RS, 0, DIM, NPH, T>(L, Rr, incP, igr, F);
        C rhoR = __shfl_down(cur.rho, 1, kWave);
        C arR[NPH > 0 ? NPH : 1];
#pragma unroll
        for (int ph = 0; ph < NPH; ++ph) arR[ph] = __shfl_down(cur.ar[ph], 1, kWave);
        face_contrib<DIM, NPH, T>(F, cur.rho, rhoR, cur.ar, arR, FCx);
#pragma unroll
        for (int q = 0; q < NF; ++q) FCl[q] = __shfl_up(FCx[q], 1, kWave);
    }
    __syncthreads();

    // ---- phase 4 ----
    double dtMin = 1.0e300;
    if (owned) {
        T Ghi[NF];
        int n = 0;
#pragma unroll
        for (int q = 0; q < NF; ++q) {
            Ghi[q] = T(0);
            if (face_slot_used<DIM, NPH, SEMI>(q)) Ghi[q] = face(n++, w, lane);
        }
        // faceArea / cellVolume
        const double vol = dxc * dyr;
        const double cx = div_fast(dyr, vol), cy = div_fast(dxc, vol);
        T acc[NF];
        accumulate<DIM, NPH, T>(acc, FCl, FCx, (T)cx, true);
        accumulate<DIM, NPH, T>(acc, Glo, Ghi, (T)cy, false);
        const double h[3] = {dxc, dyr, 1.0};
        dtMin = finish_cell<DIM, NPH, SEMI, T, SRC, C>(P, cell_index(g, col, r, 0), acc, cur, h, dt,
                                                       P.dtPartial != nullptr, raw.U, U0v);
    }
    if (P.dtPartial) {
        const double m = wave_min(dtMin);
        if (lane == 0) shMin[w] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            double b = shMin[0];
#pragma unroll
            for (int q = 1; q < NW; ++q) b = dmin_ref(b, shMin[q]);
            P.dtPartial[blockIdx.x] = b;
        }
    }
}

}  // namespace sifv
