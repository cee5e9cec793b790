// sifv_igr.hpp - information geometric regularisation (IGR) on the GPU:
// the entropic pressure sigma solves
//     sigma/rho - alpha div(grad(sigma)/rho) = alpha [tr((grad u)^2) + tr(grad u)^2]
// by in-place lexicographic Gauss-Seidel sweeps with a scalar ghost refresh
// after each sweep (IGRSolver::solveEntropicPressure, src/IGR.cpp:37-158;
// computeIGRRhs :18-35; velocity gradients src/ExplicitSolver.cpp:215-267).
//
// igr_pre_kernel   per interior cell: the right-hand side from the central
//                  velocity gradients, the diagonal (1/rho + sum of face
//                  terms) and rho itself, all from the stage's conservative
//                  buffer through the ghost mapping.
// igr_sweep_kernel the Gauss-Seidel sweeps of one solve in exactly the
//                  reference's order.
//                  Cell (i,j,k) needs the new values of (i-1,j,k), (i,j-1,k),
//                  (i,j,k-1) and the old values of the +1 neighbours, so the
//                  sweep is a wavefront.  The domain is cut into tiles of 64
//                  columns x tj (<= kIgrTj) rows of one plane; a wave owns a
//                  tile and walks its anti-diagonals (lane l <-> column, row =
//                  step - l: the left neighbour's new value comes from lane
//                  l-1's previous step, the lower neighbour's from the lane's
//                  own previous step).  Before the walk the wave stages in LDS
//                  every operand that does not depend on this sweep's new
//                  values (face densities, the old +x/+y quotients, rhs,
//                  diagonal) -- before it waits for its upstream tiles -- and,
//                  after the wait, the new values of the left column, the row
//                  below and the plane below, so the walk's dependent chain
//                  touches LDS only.  All the sweeps of a solve run in one
//                  launch, pipelined: work item (s, tile) starts when the
//                  tile's three upstream tiles have finished sweep s, the
//                  tile itself and its three downstream tiles sweep s-1, and,
//                  on a periodic axis, the far-end tile of its line sweep s-1
//                  (each tile publishes its finished sweep count in a flag
//                  array).  Boundary tiles keep the 1-deep scalar ghosts as the
//                  reference's fill after every sweep leaves them: a zero-
//                  gradient ghost is written by the tile that owns its source
//                  cell as it computes it; on a periodic axis the high tile
//                  writes the low ghost as it computes it and the low tile
//                  writes its new values into the parity slot of a side array
//                  that the high tile reads in the next sweep.  Every block
//                  takes work items in (sweep, topological tile) order and the
//                  grid never exceeds the
//                  co-resident block count; every dependency is on an earlier
//                  item, so the lowest unfinished item can always proceed.
//                  Waits are bounded: a wait that exceeds its budget raises an
//                  error flag and every wave exits.
#pragma once

#include "sifv_stage.hpp"

namespace sifv {

template <typename T>
struct IgrPreArgs {
    StageParams<T> P;   // grid, EOS, mixture, source buffer (P.src), total
    double alpha;
    double* rhs;
    double* diag;
    double* rho;        // padded; interior written here, ghosts by the scalar fill
};

template <int DIM, int NPH, typename T>
__global__ void __launch_bounds__(256) igr_pre_kernel(IgrPreArgs<T> A) {
    const StageParams<T>& P = A.P;
    const Grid& g = P.g;
    const size_t n = (size_t)g.nx * g.ny * g.nz;
    const double alpha = A.alpha;
    int i, j, k;
    for (InteriorIter it_(g.nx, g.ny, g.nz); it_.next(i, j, k);) {
        const size_t id = cell_index(g, i, j, k);
        Cell<DIM, NPH> c, m, p;
        load_cell<DIM, NPH>(P, P.src, i, j, k, c);
        // velocity gradient g[a][b] = du_a/dx_b (central, PRIM ghosts)
        double G[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
        double rhoM[3], rhoP[3];
        const double h[3] = {g.dxw[i + g.ngx], DIM >= 2 ? g.dyw[j + g.ngy] : 1.0, DIM >= 3 ? g.dzw[k + g.ngz] : 1.0};
#pragma unroll
        for (int b = 0; b < DIM; ++b) {
            load_cell<DIM, NPH>(P, P.src, i - (b == 0), j - (b == 1), k - (b == 2), m);
            load_cell<DIM, NPH>(P, P.src, i + (b == 0), j + (b == 1), k + (b == 2), p);
            const double inv = 0.5 / h[b];
#pragma unroll
            for (int a = 0; a < DIM; ++a) G[a][b] = (p.u[a] - m.u[a]) * inv;
            rhoM[b] = m.rho;
            rhoP[b] = p.rho;
        }
        double trSq = 0.0;
#pragma unroll
        for (int a = 0; a < DIM; ++a)
#pragma unroll
            for (int b = 0; b < DIM; ++b) trSq += G[a][b] * G[b][a];
        double tr = 0.0;
#pragma unroll
        for (int a = 0; a < DIM; ++a) tr += G[a][a];
        tr *= tr;
        A.rhs[id] = alpha * (trSq + tr);
        const double ri = c.rho;
        double diag = 1.0 / ri;
#pragma unroll
        for (int b = 0; b < DIM; ++b) {
            const double fl = 0.5 * (ri + rhoM[b]), fr = 0.5 * (ri + rhoP[b]);
            const double d2 = 1.0 / (h[b] * h[b]);
            diag += alpha * d2 * (1.0 / fl + 1.0 / fr);
        }
        A.diag[id] = diag;
        A.rho[id] = ri;
    }
}

struct IgrSweepArgs {
    Grid g;
    double* sg;           // sigma, padded; ghosts hold the previous sweep's fill
    const double* rho;    // padded, 1-deep ghosts by the scalar rule
    const double* rhs;
    const double* diag;
    double alpha;
    int ntx, nty, tj;     // tiles: ntx x nty x nz
    int ntiles;
    const int* order;     // tile ids in topological (anti-diagonal) order
    int* flags;           // per tile: sweeps finished (cumulative over launches)
    int epoch;            // flag value of every tile when the launch starts
    int nsweeps;          // sweeps run by this launch
    int* err;             // set when a wait exceeds its budget
    int* next;            // work-item counter, zero at launch (SIFV_IGR_DYN)
    // wrapping high faces: the first cells of each line as the previous sweep
    // left them, two slots by sweep parity ([2][nz][ny], [2][nz][nx], [2][ny][nx])
    double* wrapX;
    double* wrapY;
    double* wrapZ;
    const int* active;    // device time-loop flag (null: always run)
};

// Flags are polled with relaxed loads and each group of waits ends in one
// acquire fence: an acquire at agent scope invalidates the XCD's L2, which an
// acquiring poll loop would do on every iteration (measured 1.8x slower).
// Blocks take work items by a fixed stride of the grid (0) or from a counter
// in item order (1; 3 % slower on the 2D vortex at 1024^2 and 2048^2).
#ifndef SIFV_IGR_DYN
#define SIFV_IGR_DYN 0
#endif

__device__ __forceinline__ void igr_acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent"); }

__device__ __forceinline__ bool igr_wait(const IgrSweepArgs& A, int t, int epoch) {
    if (t < 0) return true;
    int spins = 0;
    while (__hip_atomic_load(&A.flags[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < epoch) {
        if (__hip_atomic_load(A.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
        if (++spins > (1 << 25)) {
            __hip_atomic_store(A.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        __builtin_amdgcn_s_sleep(8);
    }
    return true;
}

constexpr int kIgrTj = 16;   // most rows per sweep tile (LDS staging)
// The walk multiplies by the staged reciprocals of the face densities and of
// the diagonal instead of dividing (one rounding per operand more, within the
// parity bars; the divisions sat on the dependent chain).
#ifndef SIFV_IGR_RCP
#define SIFV_IGR_RCP 1
#endif

template <int DIM>
__global__ void __launch_bounds__(64) igr_sweep_kernel(IgrSweepArgs A) {
    if (A.active && *A.active == 0) return;
    // per-cell operands of the tile, [row][lane]
    __shared__ double sFl[kIgrTj][kWave];    // x face density to the left
    __shared__ double sTx[kIgrTj][kWave];    // old sigma(+x) / right face density
    __shared__ double sFly[DIM >= 2 ? kIgrTj : 1][kWave];
    __shared__ double sTy[DIM >= 2 ? kIgrTj : 1][kWave];
    __shared__ double sQz[DIM >= 3 ? kIgrTj : 1][kWave];   // both z quotients
    __shared__ double sRhs[kIgrTj][kWave];
    __shared__ double sDiag[kIgrTj][kWave];
    __shared__ double sLeft[kIgrTj];         // new sigma of the column left of the tile
    __shared__ double sBot[kWave];           // new sigma of the row below the tile
    __shared__ double sD2y[kIgrTj];
    const Grid& g = A.g;
    const int lane = threadIdx.x;
    const size_t sy = (size_t)g.nxT, sz = (size_t)g.nxT * g.nyT;
    const double alpha = A.alpha;
    const int ntz = DIM >= 3 ? g.nz : 1;
    const int plane = A.ntx * A.nty;
    // per face: does the scalar fill wrap (ghost from the far end of the line)?
    const bool loX = g.sbc[0] == BK_WRAP, hiX = g.sbc[1] == BK_WRAP;
    const bool loY = DIM >= 2 && g.sbc[2] == BK_WRAP, hiY = DIM >= 2 && g.sbc[3] == BK_WRAP;
    const bool loZ = DIM >= 3 && g.sbc[4] == BK_WRAP, hiZ = DIM >= 3 && g.sbc[5] == BK_WRAP;
    const int nitems = A.nsweeps * A.ntiles;
#if SIFV_IGR_DYN
    for (;;) {
        // every lane takes part in the grab (lane 0 adds 1, the others 0) and
        // in the flag store below: no lane-dependent branch may separate one
        // item from the next, or the compiler may run the lanes' loops apart
        // and read the item from a lane that did not take it
        const int q = __builtin_amdgcn_readfirstlane(
            __hip_atomic_fetch_add(A.next, lane == 0 ? 1 : 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (q >= nitems) break;
#else
    for (int q = blockIdx.x; q < nitems; q += gridDim.x) {
#endif
        const int sw = q / A.ntiles;
        const int t = A.order[q - sw * A.ntiles];
        const int I = t % A.ntx;
        const int rest = t / A.ntx;
        const int J = rest % A.nty;
        const int K = rest / A.nty;
        const int i0 = I * kWave;
        const int i = i0 + lane;
        const int j0 = J * A.tj;
        const int nrows = (j0 + A.tj <= g.ny) ? A.tj : g.ny - j0;
        const bool colOk = i < g.nx;
        const int ci = colOk ? i : g.nx - 1;
        const double dx = g.dxw[ci + g.ngx];
        const double d2x = 1.0 / (dx * dx);
        const double d2z = DIM >= 3 ? 1.0 / (g.dzw[K + g.ngz] * g.dzw[K + g.ngz]) : 0.0;
        const int now = A.epoch + sw + 1, prev = A.epoch + sw;
        // sweep sw > 0 follows the tile's own sweep sw-1 (another block may
        // have run it), reads the downstream tiles' values of sweep sw-1, and a
        // low tile on a wrapping axis replaces the high ghost the far-end tile
        // read in sweep sw-1 (sweep 0 is ordered by the launch itself)
        bool ok = true;
        if (sw > 0) {
            ok = igr_wait(A, t, prev);
            ok = ok && igr_wait(A, I < A.ntx - 1 ? t + 1 : -1, prev);
            ok = ok && igr_wait(A, DIM >= 2 && J < A.nty - 1 ? t + A.ntx : -1, prev);
            ok = ok && igr_wait(A, DIM >= 3 && K < ntz - 1 ? t + plane : -1, prev);
            ok = ok && igr_wait(A, (loX || hiX) && I == 0 && A.ntx > 1 ? t + A.ntx - 1 : -1, prev);
            ok = ok && igr_wait(A, (loY || hiY) && J == 0 && A.nty > 1 ? t + (A.nty - 1) * A.ntx : -1, prev);
            ok = ok && igr_wait(A, (loZ || hiZ) && K == 0 && ntz > 1 ? t + (ntz - 1) * plane : -1, prev);
            if (!ok) return;
            igr_acquire();
        }
        // wrapping high faces read the first cells of the line as the previous
        // sweep left them: from the ghost the fill before the launch wrote, and
        // later from the side slot the low tile filled in sweep sw-1
        const int par = (A.epoch + sw) & 1, npar = par ^ 1;
        // operands that this sweep's new values do not change: the +x / +y
        // neighbours are in this tile or in tiles that wait for it
#pragma unroll 4
        for (int jj = 0; jj < kIgrTj; ++jj) {
            if (jj < nrows && colOk) {
                const size_t id = cell_index(g, i, j0 + jj, K);
                const double ri = A.rho[id];
#if SIFV_IGR_RCP
                sFl[jj][lane] = 1.0 / (0.5 * (ri + A.rho[id - 1]));
#else
                sFl[jj][lane] = 0.5 * (ri + A.rho[id - 1]);
#endif
                double sr = A.sg[id + 1];
                if (hiX && sw > 0 && i == g.nx - 1) sr = A.wrapX[((size_t)par * ntz + K) * g.ny + j0 + jj];
                sTx[jj][lane] = sr / (0.5 * (ri + A.rho[id + 1]));
                if (DIM >= 2) {
#if SIFV_IGR_RCP
                    sFly[jj][lane] = 1.0 / (0.5 * (ri + A.rho[id - sy]));
#else
                    sFly[jj][lane] = 0.5 * (ri + A.rho[id - sy]);
#endif
                    double st = A.sg[id + sy];
                    if (hiY && sw > 0 && j0 + jj == g.ny - 1) st = A.wrapY[((size_t)par * ntz + K) * g.nx + i];
                    sTy[jj][lane] = st / (0.5 * (ri + A.rho[id + sy]));
                }
                sRhs[jj][lane] = A.rhs[id];
#if SIFV_IGR_RCP
                sDiag[jj][lane] = 1.0 / A.diag[id];
#else
                sDiag[jj][lane] = A.diag[id];
#endif
            }
        }
        if (DIM >= 2 && lane < nrows) {
            const double hy = g.dyw[j0 + lane + g.ngy];
            sD2y[lane] = 1.0 / (hy * hy);
        }
        ok = igr_wait(A, I > 0 ? t - 1 : -1, now);
        ok = ok && igr_wait(A, DIM >= 2 && J > 0 ? t - A.ntx : -1, now);
        ok = ok && igr_wait(A, DIM >= 3 && K > 0 ? t - plane : -1, now);
        if (!ok) return;
        igr_acquire();
        // new values published by the upstream tiles (ghosts at domain edges)
        if (lane < nrows) sLeft[lane] = A.sg[cell_index(g, i0 - 1, j0 + lane, K)];
        if (DIM >= 2 && colOk) sBot[lane] = A.sg[cell_index(g, i, j0 - 1, K)];
        if (DIM >= 3) {
#pragma unroll 4
            for (int jj = 0; jj < kIgrTj; ++jj) {
                if (jj < nrows && colOk) {
                    const size_t id = cell_index(g, i, j0 + jj, K);
                    const double ri = A.rho[id];
                    const double fl = 0.5 * (ri + A.rho[id - sz]), fr = 0.5 * (ri + A.rho[id + sz]);
                    double su = A.sg[id + sz];
                    if (hiZ && sw > 0 && K == g.nz - 1) su = A.wrapZ[((size_t)par * g.ny + j0 + jj) * g.nx + i];
                    sQz[jj][lane] = A.sg[id - sz] / fl + su / fr;
                }
            }
        }
        __syncthreads();
        double last = 0.0;
        for (int s = 0; s < nrows + kWave - 1; ++s) {
            const int jj = s - lane;
            const double fromLeft = __shfl_up(last, 1);
            if (colOk && jj >= 0 && jj < nrows) {
                double off = 0.0;
                {
                    const double sl = lane == 0 ? sLeft[jj] : fromLeft;
#if SIFV_IGR_RCP
                    off += alpha * d2x * (sl * sFl[jj][lane] + sTx[jj][lane]);
#else
                    off += alpha * d2x * (sl / sFl[jj][lane] + sTx[jj][lane]);
#endif
                }
                if (DIM >= 2) {
                    const double sl = jj == 0 ? sBot[lane] : last;
#if SIFV_IGR_RCP
                    off += alpha * sD2y[jj] * (sl * sFly[jj][lane] + sTy[jj][lane]);
#else
                    off += alpha * sD2y[jj] * (sl / sFly[jj][lane] + sTy[jj][lane]);
#endif
                }
                if (DIM >= 3) off += alpha * d2z * sQz[jj][lane];
#if SIFV_IGR_RCP
                last = (sRhs[jj][lane] + off) * sDiag[jj][lane];
#else
                last = (sRhs[jj][lane] + off) / sDiag[jj][lane];
#endif
                const size_t id = cell_index(g, i, j0 + jj, K);
                A.sg[id] = last;
                // ghosts of the boundary cells as the scalar fill after this
                // sweep leaves them: zero-gradient ghosts copy the cell, the
                // low ghost of a periodic axis the last cell of the line
                if (i == 0) {
                    if (!loX) A.sg[id - 1] = last;
                    if (hiX) A.wrapX[((size_t)npar * ntz + K) * g.ny + j0 + jj] = last;
                }
                if (i == g.nx - 1) {
                    if (loX) A.sg[id - (size_t)g.nx] = last;
                    if (!hiX) A.sg[id + 1] = last;
                }
                if (DIM >= 2) {
                    const int j = j0 + jj;
                    if (j == 0) {
                        if (!loY) A.sg[id - sy] = last;
                        if (hiY) A.wrapY[((size_t)npar * ntz + K) * g.nx + i] = last;
                    }
                    if (j == g.ny - 1) {
                        if (loY) A.sg[id - (size_t)g.ny * sy] = last;
                        if (!hiY) A.sg[id + sy] = last;
                    }
                }
                if (DIM >= 3) {
                    if (K == 0) {
                        if (!loZ) A.sg[id - sz] = last;
                        if (hiZ) A.wrapZ[((size_t)npar * g.ny + j0 + jj) * g.nx + i] = last;
                    }
                    if (K == g.nz - 1) {
                        if (loZ) A.sg[id - (size_t)g.nz * sz] = last;
                        if (!hiZ) A.sg[id + sz] = last;
                    }
                }
            }
        }
        // publish the tile: data before flag (every lane stores the same value)
        __threadfence();
        __syncthreads();
        __hip_atomic_store(&A.flags[t], now, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------------------
// Strip-streaming sweep (2D).  A wave owns a strip of 64 columns and walks
// every row of every sweep of the solve: at schedule step s lane l updates
// row r = s - l, where r runs over the sweeps with period P = ny + gap (rows
// ny..P-1 of a period are idle).  The left neighbour's new value is lane
// l-1's result of the previous step (DPP shift), the lower one the lane's
// own previous result, the +x neighbour's old value is what lane l+1 holds
// as its +y operand (DPP shift), so no tile waits for another tile to finish.
// Per cell the pack kernel stores the five coefficients of the update
//     new = c0 + cR*right + cT*top + cB*bottom + cL*left,
// c0 = rhs/diag, cX = alpha/h^2 / rho_face / diag, and sigma, in a cyclic
// skew: cell (l, j) of a strip sits in slot (j + l) mod ns, P a multiple of ns, so
// at step s every lane reads slot s mod ns whatever row and sweep it is at: one
// contiguous slot of 64 x 6 doubles (three 16-byte loads per lane).  Lane
// 0's left values and the last lane's right values cross strips through edge
// arrays (by sweep parity), handed over per group of kStripGroup steps.  On a
// wrapping x axis sweep q of strip 0 needs sweep q-1 of the last strip on the same
// row, while each strip trails its left neighbour by 64 steps and more: the gap
// between sweeps makes room for that skew (strip_period(): 64 W + 64 + 32 steps, 72
// more than the dependencies need).
// What bounds it: the serial chain of a group (8 steps of two dependent multiply-
// adds and a shift, with the LDS reads and counters around them about 0.65 us)
// times (ny + 64 W) / 8, and around a wrapping axis the hand-off of every strip
// (about 8 us beyond the 64 steps).  Microseconds a sweep, one wave with loads,
// coefficients and sweeps in one and a release / acquire hand-off -> now: 1024^2
// wrapping 468 -> 242, 1024^2 walls 240 -> 144, 2048^2 981 -> 521 and 580 -> 318.
// Ghost semantics are those of the per-sweep scalar fill: zero-gradient
// faces read the cell's own previous-sweep value, wrapping y faces the
// previous result (bottom) and the saved previous-sweep row-0 value (top).
constexpr int kStripGroup = 8;     // steps per group: of loads, of computation, of hand-off
constexpr int kStripMinRows = 152; // lane skew, prefetched steps and a margin: a sweep's records are written before they are read again
// A record slot (doubles): three arrays of 64 pairs, (c0, cR), (cT, sigma
// of the cell in the next slot, that is of the row above), (cB, cL), so each of a
// step's three 16-byte loads per lane is one contiguous KB (with the six values of
// a lane adjacent every load touched all 24 lines of the slot), and a step needs
// nothing of the next one's records (with a cell's own sigma in its slot the +y
// operand of a group's last step waited for the next group, halving the distance
// of the loads ahead); the cell's own old value is the step before's +y operand.
constexpr int kStripSlot = 6 * kWave;
__device__ __forceinline__ size_t strip_sigma(int lane) { return 2 * kWave + 2 * (size_t)lane + 1; }

// An edge value handed from strip to strip: two 64-bit words, each half of the
// value beside the tag of the sweep it belongs to, stored and loaded at device
// scope (past the XCDs' L2s).  A reader polls the words themselves: no fence, which
// would write back or invalidate an L2 shared by other strips, and no progress
// flag, whose store has to wait for the values' and whose poll is one more round
// trip (1024^2 wrapping: 330 us a sweep, with fences and flags 356).
__device__ __forceinline__ void edge_store(unsigned long long* p, double v, unsigned tag) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v), t = (unsigned long long)tag << 32;
    __hip_atomic_store(p, t | (b & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p + 1, t | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool edge_load(const unsigned long long* p, unsigned tag, double& v) {
    const unsigned long long a = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long b = __hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = __longlong_as_double((long long)((b << 32) | (a & 0xffffffffull)));
    return (unsigned)(a >> 32) == tag && (unsigned)(b >> 32) == tag;
}

struct IgrStripPackArgs {
    Grid g;
    const double* sigma;   // padded
    const double* rho;     // padded, ghosts filled
    const double* rhs;
    const double* diag;
    double alpha;
    double* rec;           // [W][ns] record slots
    unsigned long long* edgeL;   // [2][W][ny][2]
    unsigned long long* edgeR;   // [2][W][ny][2]
    unsigned tag;          // of the initial iterate's edge values
    int W;
    int ns;                // slots per strip
};

// Threads run in record order (strip, slot, lane): each wave writes one
// contiguous 3 KB slot, and reads the slot's diagonal of cells (row = slot -
// lane), whose lines the neighbouring slots share in L2.
template <int DIM>
__global__ void __launch_bounds__(256) igr_strip_pack_kernel(IgrStripPackArgs A) {
    const Grid& g = A.g;
    const size_t sy = (size_t)g.nxT;
    const size_t total = (size_t)A.W * A.ns * kWave;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
        const int l = (int)(e % kWave);
        const size_t ws = e / kWave;
        const int t = (int)(ws % A.ns), w = (int)(ws / A.ns);
        const int i = w * kWave + l;
        if (i >= g.nx) continue;
        int j = t - l;
        if (j < 0) j += A.ns;
        double2* r = reinterpret_cast<double2*>(A.rec + ws * kStripSlot) + l;
        if (j >= g.ny) {
            // the gap slot before row 0 holds row 0's sigma
            if (j == A.ns - 1) r[kWave].y = A.sigma[cell_index(g, i, 0, 0)];
            continue;
        }
        const size_t id = cell_index(g, i, j, 0);
        const double ri = A.rho[id];
        const double rd = 1.0 / A.diag[id];
        const double hx = g.dxw[i + g.ngx], hy = g.dyw[j + g.ngy];
        const double ax = A.alpha / (hx * hx), ay = A.alpha / (hy * hy);
        const double sg = A.sigma[id];
        // the row above; above the last row only when the slots wrap there
        const double up = A.sigma[cell_index(g, i, j + 1 < g.ny ? j + 1 : 0, 0)];
        r[0] = make_double2(A.rhs[id] * rd, ax / (0.5 * (ri + A.rho[id + 1])) * rd);
        r[kWave] = make_double2(ay / (0.5 * (ri + A.rho[id + sy])) * rd, up);
        r[2 * kWave] = make_double2(ay / (0.5 * (ri + A.rho[id - sy])) * rd, ax / (0.5 * (ri + A.rho[id - 1])) * rd);
        // edge values of "sweep -1" (parity slot 1): the initial iterate
        const int L = min(kWave - 1, g.nx - 1 - w * kWave);
        if (l == 0) edge_store(A.edgeL + 2 * (((size_t)A.W + w) * g.ny + j), sg, A.tag);
        if (l == L) edge_store(A.edgeR + 2 * (((size_t)A.W + w) * g.ny + j), sg, A.tag);
    }
}

template <int DIM>
__global__ void __launch_bounds__(256) igr_strip_unpack_kernel(Grid g, const double* rec, double* sigma, int ns) {
    int i, j, k;
    for (InteriorIter it_(g.nx, g.ny, 1); it_.next(i, j, k);) {
        const int w = i / kWave, l = i - w * kWave;
        int t = j + l - 1;
        t = t < 0 ? t + ns : t >= ns ? t - ns : t;
        sigma[cell_index(g, i, j, 0)] = rec[((size_t)w * ns + t) * kStripSlot + strip_sigma(l)];
    }
}

struct IgrStripArgs {
    int nx, ny;
    double* rec;
    unsigned long long* edgeL;
    unsigned long long* edgeR;
    unsigned tag;          // of the initial iterate's edge values; sweep q's carry tag + q + 1
    int* err;
    const int* active;
    int W, P, nsweeps;
    int ns;                // record slots per strip; P is a multiple of it
    int perX, perY;
    long long waitTicks;   // longest wait, in ticks of the device's wall clock
};

__device__ __forceinline__ double dpp_shl1(double v) {   // lane l <- lane l+1
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x130, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x130, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// The same shifts with the lane that has no source (0 / 63) taking edge's value.
__device__ __forceinline__ double dpp_shr1_in(double v, double edge) {
    const long long b = __double_as_longlong(v), e = __double_as_longlong(edge);
    const int lo = __builtin_amdgcn_update_dpp((int)e, (int)b, 0x138, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(e >> 32), (int)(b >> 32), 0x138, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double dpp_shl1_in(double v, double edge) {
    const long long b = __double_as_longlong(v), e = __double_as_longlong(edge);
    const int lo = __builtin_amdgcn_update_dpp((int)e, (int)b, 0x130, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(e >> 32), (int)(b >> 32), 0x130, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// Seven waves per strip, one duty each, so that the serial chain holds nothing
// that does not depend on it and the duties' round trips do not add up:
//   wave 0 carries the sweeps: new = base + cB*bottom + cL*left;
//   waves 1 and 2 bring the records (even and odd groups), two groups each in
//     registers on their way from memory and up to kStripRecGroups in LDS;
//   wave 3 works out base = c0 + cR*right + cT*top, which has previous-sweep
//     values only, in place of c0 in the LDS record;
//   wave 4 publishes the edge values of the groups wave 0 finishes;
//   waves 5 and 6 poll the left and the right neighbour's edge values of upcoming
//     groups, up to kStripRing steps ahead.
// The sigma that wave 0 stores into a record is read again P steps later (slots that
// come round sooner belong to idle rows, whose values nothing uses).  That record is
// loaded at most kStripRecGroups + 4 groups ahead of the groups counted as done, and
// wave 0 counts a group as done with the stores of at most kStripStoreGroups groups
// outstanding (waiting for all but two groups made the stores' latency the limit), so
// the store is complete if the steps of a period that store anything, ny or more and
// so at least kStripMinRows, exceed all of them together.
// Every wait is bounded, by time (strips may wait for CUs that another stream's
// kernels hold, and a pass of a wave that polls LDS is some 50 ns), and ends on the
// abort flag.
constexpr int kStripRecGroups = 5;
constexpr int kStripStoreGroups = 7;
static_assert(kStripMinRows > kStripGroup * (kStripRecGroups + 4 + kStripStoreGroups), "a store before its reload");
static_assert(kStripGroup * kStripStoreGroups <= 63, "the counter of vector memory operations has 6 bits");
constexpr int kStripWaves = 7;
constexpr int kStripRing = 192;   // steps of wave 0's results and inputs held in LDS

template <int DIM>
__global__ void __launch_bounds__(64 * kStripWaves) igr_strip_kernel(IgrStripArgs A) {
    if (A.active && *A.active == 0) return;
    constexpr int U = kStripGroup, RS = kStripRing, RG = kStripRecGroups;
    static_assert(RS % U == 0 && RS >= 2 * kWave, "whole groups; helpers move up to a wave of steps at once");
    __shared__ __align__(16) double sIn[2][RS];  // neighbours' values: [left/right][step mod RS]
    __shared__ double sOut[RS][2];               // wave 0's results of lanes 0 and L: [step mod RS]
    __shared__ double2 sRec[RG * U][3][kWave];   // records: [step mod RG U]
    // groups: [0] left inputs loaded, [1] right inputs loaded, [2] published,
    // [3] abort, [4] done by wave 0, [5], [6] even / odd record groups loaded,
    // [7] bases worked out
    __shared__ int sFlag[8];
    const int w = blockIdx.x, lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);   // wave-uniform
    const int ny = A.ny, P = A.P, W = A.W, ns = A.ns;
    const int L = min(kWave - 1, A.nx - 1 - w * kWave);
    const int Rt = A.nsweeps * P;
    const int nsteps = Rt + kWave - 1;
    const int ngroups = (nsteps + U - 1) / U;
    const bool leftWall = w == 0 && !A.perX, rightWall = w == W - 1 && !A.perX;
    const int leftSrc = w > 0 ? w - 1 : W - 1, rightSrc = w < W - 1 ? w + 1 : 0;
    double* rec = A.rec + (size_t)w * ns * kStripSlot;
    if (threadIdx.x < 8) sFlag[threadIdx.x] = 0;
    __syncthreads();
    auto lds_load = [](int* p) __attribute__((always_inline)) { return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP); };
    auto lds_store = [](int* p, int v) __attribute__((always_inline)) { __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP); };
    // the helper waves watch the device error flag and raise the block's abort
    // flag, which waves 0 and 3 poll in LDS
    auto aborted = [&]() __attribute__((always_inline)) { return __hip_atomic_load(&sFlag[3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0; };
    // true when a wait whose first look was at `since` has been too long
    auto late = [&](int looks, long long& since) __attribute__((always_inline)) {
        const long long t = wall_clock64();
        if (looks == 1) since = t;
        return t - since > A.waitTicks;
    };
    // one idle pass of a helper wave (idle: passes since it last moved); true: give up
    long long since = 0;
    auto idle_pass = [&](int& idle) __attribute__((always_inline)) {
        bool stop = aborted();
        if ((++idle & 255) == 0) {
            if (late(idle >> 8, since)) __hip_atomic_store(A.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            stop = stop || __hip_atomic_load(A.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        }
        if (stop) __hip_atomic_store(&sFlag[3], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return stop;
    };
    if (wave == 4) {
        int pub = 0, idle = 0;
        while (pub < ngroups) {
            const int done = min(lds_load(&sFlag[4]), pub + kWave / U);
            if (done == pub) {
                if (idle_pass(idle)) return;
                continue;
            }
            idle = 0;
            const int s = pub * U + lane;
            const bool in = s < done * U;
            const double* o = sOut[s % RS];
            int r = s;
            bool v = in && r < Rt && r % P < ny;
            if (v) edge_store(A.edgeL + 2 * (((size_t)((r / P) & 1) * W + w) * ny + r % P), o[0], A.tag + r / P + 1);
            r = s - L;
            v = in && r >= 0 && r < Rt && r % P < ny;
            if (v)
                edge_store(A.edgeR + 2 * (((size_t)((r / P) & 1) * W + w) * ny + r % P), o[L > 0 ? 1 : 0],
                           A.tag + r / P + 1);
            lds_store(&sFlag[2], done);
            pub = done;
        }
        return;
    }
    if (wave == 1 || wave == 2) {
        const int odd = wave - 1;
        double ra[6][U], rb[6][U];
        int tp = odd * U % ns;   // slot of the next step loaded
        auto load = [&](double (&r)[6][U]) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const double2* p = reinterpret_cast<const double2*>(rec + (size_t)tp * kStripSlot) + lane;
#pragma unroll
                for (int f = 0; f < 3; ++f) {
                    const double2 v = p[f * kWave];
                    r[2 * f][k] = v.x;
                    r[2 * f + 1][k] = v.y;
                }
                if (++tp == ns) tp = 0;
            }
            tp = (tp + U) % ns;
        };
        int idle = 0;
        auto put = [&](int g, const double (&r)[6][U]) __attribute__((always_inline)) {
            while (lds_load(&sFlag[4]) + RG <= g)
                if (idle_pass(idle)) return false;
            idle = 0;
#pragma unroll
            for (int k = 0; k < U; ++k)
#pragma unroll
                for (int f = 0; f < 3; ++f)
                    sRec[g % RG * U + k][f][lane] = make_double2(r[2 * f][k], r[2 * f + 1][k]);
            lds_store(&sFlag[5 + odd], g + 1);
            return true;
        };
        load(ra);
        load(rb);
        for (int g = odd; g < ngroups; g += 4) {
            if (!put(g, ra)) return;
            load(ra);
            if (g + 2 >= ngroups) return;
            if (!put(g + 2, rb)) return;
            load(rb);
        }
        return;
    }
    if (wave >= 5) {
        const bool right = wave == 6;
        int* loadedFlag = &sFlag[right ? 1 : 0];
        if (right ? rightWall : leftWall) {
            lds_store(loadedFlag, ngroups);
            return;
        }
        const int src = right ? rightSrc : leftSrc;
        const unsigned long long* edges = right ? A.edgeL : A.edgeR;
        const int back = !right && w > 0 ? 0 : 1;   // sweeps back
        int loaded = 0, idle = 0;
        int span = 1;   // groups polled at once: one while waiting, so that the polls leave the memory to others
        while (loaded < ngroups) {
            // slots of groups wave 0 has finished are free again
            const int upto = min(min(ngroups, lds_load(&sFlag[4]) + RS / U), loaded + span);
            // lane m polls the value of step loaded U + m: the row of lane 0 (left)
            // or of the last lane (right)
            const int s = loaded * U + lane;
            const int r = s - (right ? L : 0);
            const bool v = s < upto * U && r >= 0 && r < Rt && r % P < ny;
            double a = 0.0;
            bool ready = s < upto * U;
            if (v) {
                const int q = r / P - back;
                ready = edge_load(edges + 2 * (((size_t)(q & 1) * W + src) * ny + r % P), A.tag + q + 1, a);
            }
            // groups whose every step is there, from the front
            const unsigned long long ok = __ballot(ready);
            const int got = (ok == ~0ull ? kWave : __builtin_ctzll(~ok)) / U;
            if (got == 0) {
                span = 1;
                if (idle_pass(idle)) return;
                continue;
            }
            span = min(2 * span, kWave / U);
            idle = 0;
            if (lane < got * U) sIn[right ? 1 : 0][s % RS] = a;
            loaded += got;
            lds_store(loadedFlag, loaded);
        }
        return;
    }
    // waves 0 and 3 read their counters together and ahead of need; see() is where
    // they are looked at, and orders what is read after it
    auto peek = [&](int f) __attribute__((always_inline)) { return __hip_atomic_load(&sFlag[f], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    auto see = [&]() __attribute__((always_inline)) { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup"); };
    const double* sig0 = rec + strip_sigma(lane);
    // (cell (lane, j)'s sigma is in slot j + lane - 1)
    const double first = sig0[(size_t)(lane > 0 ? lane - 1 : ns - 1) * kStripSlot];   // row 0 of the initial iterate
    if (wave == 3) {
        // row 0 of the previous sweep; +y operand of the step before (the cell's own
        // old value); row in the period of the lane's next step
        double row0 = first, above = sig0[(size_t)(ns - 1) * kStripSlot];
        int jc = lane == 0 ? 0 : P - lane;
        // the period's row of lane 63 at the group's first step, slot of the group
        int pos = P - (kWave - 1), r0 = 0, i0 = 0;
        int inR = 0, recs[2] = {0, 0}, idle = 0;
        auto bases = [&](int g, int odd) __attribute__((always_inline)) {
            while (recs[odd] <= g || inR <= g) {
                const int e = peek(5), o = peek(6), n = peek(1), ab = peek(3);
                recs[0] = __builtin_amdgcn_readfirstlane(e);
                recs[1] = __builtin_amdgcn_readfirstlane(o);
                inR = __builtin_amdgcn_readfirstlane(n);
                if (recs[odd] > g && inR > g) break;
                if (__builtin_amdgcn_readfirstlane(ab) != 0 || idle_pass(idle)) return false;
            }
            see();
            idle = 0;
            double2 cr[U], ct[U];
            double rv[U];
#pragma unroll
            for (int k = 0; k < U; ++k) {
                rv[k] = sIn[1][i0 + k];
                cr[k] = sRec[r0 + k][0][lane];
                ct[k] = sRec[r0 + k][1][lane];
            }
            if (leftWall && lane == 0) {
                // beyond the wall: the cell's own old value
#pragma unroll
                for (int k = 0; k < U; ++k) sIn[0][i0 + k] = k > 0 ? ct[k > 0 ? k - 1 : 0].y : above;
            }
            if (pos >= 1 && pos + kWave + U - 2 <= ny - 2 && L == kWave - 1) {
                // every lane at an interior row, and the neighbour's value comes in at
                // the lane without a source of the shift
                if (rightWall) {
#pragma unroll
                    for (int k = 0; k < U; ++k) rv[k] = k > 0 ? ct[k > 0 ? k - 1 : 0].y : above;
                }
#pragma unroll
                for (int k = 0; k < U; ++k) {
                    const double right = dpp_shl1_in(ct[k].y, rv[k]);
                    sRec[r0 + k][0][lane].x = cr[k].x + cr[k].y * right + ct[k].x * ct[k].y;
                }
                above = ct[U - 1].y;
                jc += U;
            } else {
#pragma unroll
                for (int k = 0; k < U; ++k) {
                    const double sgT = ct[k].y, cellOld = above;
                    above = sgT;
                    const double top = jc < ny - 1 ? sgT : (A.perY ? row0 : cellOld);
                    const double rightS = dpp_shl1(sgT);
                    const double right = lane < L ? rightS : (rightWall ? cellOld : rv[k]);
                    sRec[r0 + k][0][lane].x = cr[k].x + cr[k].y * right + ct[k].x * top;
                    // at a period's end the slot holds the sweep's own row 0
                    if (++jc == P) {
                        row0 = sgT;
                        jc = 0;
                    }
                }
            }
            lds_store(&sFlag[7], g + 1);
            if ((pos += U) >= P) pos -= P;
            if ((r0 += U) == RG * U) r0 = 0;
            if ((i0 += U) == RS) i0 = 0;
            return true;
        };
        for (int g = 0; g < ngroups; g += 2) {
            if (!bases(g, 0)) return;
            if (g + 1 < ngroups && !bases(g + 1, 1)) return;
        }
        return;
    }
    // wave 0: the sweeps
    __builtin_amdgcn_s_setprio(3);
    const bool act = lane <= L;
    double* sig = rec + strip_sigma(lane);
    // lane state: row 0 of the previous sweep, last result
    double row0 = first;
    int tl = ny - 2 + lane;
    if (tl >= ns) tl -= ns;
    double last = A.perY ? sig[(size_t)tl * kStripSlot] : row0;
    // row in the period of the lane's next step, and of lane 63's at the group's
    // first; slot the next step's result goes to; places of the group in the rings
    int jc = lane == 0 ? 0 : P - lane;
    int pos = P - (kWave - 1), tc = ns - 1, r1 = 0, i0 = 0;
    // the lanes whose results the neighbours read
    const bool edge = lane == 0 || lane == L;
    const int edgeCol = lane == 0 ? 0 : 1;
    double base[2][U];
    double2 cbl[2][U];
    // left inputs and bases of a group there, and its output slots published by wave
    // 4: the counters last seen
    int inL = 0, pub = 0, done3 = 0, spins = 0;
    auto count = [&](int l, int d, int p) __attribute__((always_inline)) {
        inL = __builtin_amdgcn_readfirstlane(l);
        done3 = __builtin_amdgcn_readfirstlane(d);
        pub = __builtin_amdgcn_readfirstlane(p);
    };
    auto wait = [&](int g, int gBase) __attribute__((always_inline)) {
        while (inL <= g || done3 <= gBase || pub <= g - RS / U) {
            const int l = peek(0), d = peek(7), p = peek(2), ab = peek(3);
            count(l, d, p);
            if (__builtin_amdgcn_readfirstlane(ab) != 0) return false;
            if ((++spins & 0xffff) == 0 && late(spins >> 16, since)) {
                __hip_atomic_store(A.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&sFlag[3], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                return false;
            }
        }
        see();
        spins = 0;
        return true;
    };
    // next group's records (after the last group: of any old one, unused)
    auto fetch = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < U; ++k) {
            base[b][k] = sRec[r1 + k][0][lane].x;
            cbl[b][k] = sRec[r1 + k][2][lane];
        }
        if ((r1 += U) == RG * U) r1 = 0;
    };
    // byte offsets of the lane's sigma in the slots of a group
    unsigned sigOff[U];
#pragma unroll
    for (int k = 0; k < U; ++k) sigOff[k] = 8 * (unsigned)(k * kStripSlot + strip_sigma(lane));
    auto group = [&](int g, int b) __attribute__((always_inline)) {
        double (*out)[2] = &sOut[i0];
        // the neighbour's values, the same in every lane; read before the next
        // group's records, behind which they would wait
        double lv[U];
        int l, d, p;
        auto read = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < U; ++k) lv[k] = sIn[0][i0 + k];
            __builtin_amdgcn_sched_barrier(0);
            fetch(1 - b);
            l = peek(0), d = peek(7), p = peek(2);
            __builtin_amdgcn_sched_barrier(0);
        };
        if (pos >= 1 && pos + kWave + U - 2 <= ny - 2 && tc + U <= ns) {
            // every lane's row is an interior row (1 .. ny-2) of one sweep: all lanes
            // update, none meets a boundary row, and all write the same record slot
            // (lanes past the mesh edge their padding records)
            read();
            char* dst = reinterpret_cast<char*>(rec + (size_t)tc * kStripSlot);
            double nw[U];
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const double left = dpp_shr1_in(last, lv[k]);
                last = nw[k] = base[b][k] + cbl[b][k].x * last + cbl[b][k].y * left;
                *reinterpret_cast<double*>(dst + sigOff[k]) = last;
            }
            if (edge) {
#pragma unroll
                for (int k = 0; k < U; ++k) out[k][edgeCol] = nw[k];
            }
            jc += U;
            if ((tc += U) == ns) tc = 0;
        } else {
            // general steps: any row position (first or last row of a sweep,
            // gap rows, rows outside the launch)
            read();
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const int s = g * U + k;
                if (s >= nsteps) break;
                const int r = s - lane;
                const bool valid = act && r >= 0 && r < Rt && jc < ny;
                const double bot = jc > 0 || A.perY ? last : row0;
                const double left = dpp_shr1_in(last, lv[k]);
                const double nw = base[b][k] + cbl[b][k].x * bot + cbl[b][k].y * left;
                if (valid) {
                    if (jc == 0) row0 = nw;
                    sig[(size_t)tc * kStripSlot] = nw;
                    last = nw;
                }
                if (edge) out[k][edgeCol] = nw;
                if (++jc == P) jc = 0;
                if (++tc == ns) tc = 0;
            }
        }
        // stores of all but the last kStripStoreGroups groups are done
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kStripGroup * kStripStoreGroups) : "memory");
        lds_store(&sFlag[4], g + 1);
        count(l, d, p);
        if ((pos += U) >= P) pos -= P;
        if ((i0 += U) == RS) i0 = 0;
    };
    if (!wait(-1, 0)) return;
    fetch(0);
    for (int g = 0; g < ngroups; g += 2) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            if (g + b >= ngroups) return;
            if (!wait(g + b, min(g + b + 1, ngroups - 1))) return;
            group(g + b, b);
        }
    }
}

}  // namespace sifv
