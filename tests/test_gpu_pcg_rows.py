"""Rows of the conjugate-gradient operator whose face weights are formed from the
densities: meshes at, one past and short of the bricks' columns, rows and planes, odd
children in the restriction, wrapping and wall faces per axis, and densities under the
floor of 1e-14 (a time step at which the floored faces' terms are of the mass term's
size).  Counts and answers against the oracle's solve to the same tolerance, 1e-7 (at
1e-9 the residual plateaus and the crossing iteration is a matter of rounding):
answers within 1e3 tol, the bar of the 2D solves, counts within max(2, 10 %)."""
import numpy as np
import pytest

from semiimplicitfv_amd import HLLCSolver, IdealGasEOS, MGPCGPressureSolver, PCGPressureSolver, SemiImplicitSolver
from tests.golden import problems

pytestmark = pytest.mark.gpu

SOLVERS = {"PCG": PCGPressureSolver, "MGPCG": MGPCGPressureSolver}
SHAPES = [((64, 8, 16), (1, 1, 1)), ((65, 9, 17), (0, 1, 0)), ((67, 5, 33), (1, 0, 0)), ((63, 7, 15), (0, 0, 0)),
          ((129, 17, 1), (1, 1, 0)), ((66, 3, 1), (0, 0, 0))]


def _system(shape, periods, floor):
    cfg, mesh, rho, rhoc2, rhs = problems.pressure_problem_nd(shape, periods, seed=3)
    dt = 0.3
    if floor:
        mesh.interior(rho)[..., ::3] = 1e-16
        rho = problems._fill_scalar_np(mesh, rho)
        hx = 1.0 / max(shape)
        dt = hx / np.sqrt(1e14 * mesh.interior(rhoc2).max())
    return cfg, mesh, rho, rhoc2, rhs, dt


@pytest.mark.parametrize("kind", ["PCG", "MGPCG"])
@pytest.mark.parametrize("floor", [False, True])
@pytest.mark.parametrize("shape,periods", SHAPES)
def test_pcg_rows_from_densities(gpu, oracle_c, shape, periods, floor, kind):
    cfg, mesh, rho, rhoc2, rhs, dt = _system(shape, periods, floor)
    tol = 1e-7
    eos = IdealGasEOS(1.4, 1.0, cfg)
    g = SemiImplicitSolver(mesh, HLLCSolver(eos), SOLVERS[kind](), eos, None, cfg)
    pg, pc = np.zeros(mesh.totalCells()), np.zeros(mesh.totalCells())
    ig = SOLVERS[kind](g).solve(mesh, rho, rhoc2, rhs, pg, dt, tol, 2000)
    g.close()
    cpu = oracle_c.CpuSolver(mesh, cfg, 2, eos, "c")
    ic = (cpu.pcg if kind == "PCG" else cpu.mgpcg)(rho, rhoc2, rhs, pc, dt, tol, 2000)
    assert 0 < ig < 2000 and abs(ig - ic) <= max(2, ic // 10), (ig, ic)
    ref = mesh.interior(pc)
    assert np.abs(mesh.interior(pg) - ref).max() <= 1e3 * tol * np.abs(ref).max()


@pytest.mark.parametrize("kind", ["PCG", "MGPCG"])
@pytest.mark.parametrize("shape,periods", [((65, 9, 17), (0, 1, 0)), ((66, 7, 1), (1, 0, 0))])
def test_pcg_infinite_density(gpu, oracle_c, shape, periods, kind):
    """Faces of a cell of infinite density have weight 0 and everything stays finite;
    the bars of test_pcg_rows_from_densities."""
    cfg, mesh, rho, rhoc2, rhs, dt = _system(shape, periods, False)
    mesh.interior(rho)[..., ::3, 5::7] = np.inf
    mesh.interior(rho)[..., 1, 11:13] = np.inf
    mesh.interior(rho)[..., 0, 0] = np.inf
    rho = problems._fill_scalar_np(mesh, rho)
    tol = 1e-7
    eos = IdealGasEOS(1.4, 1.0, cfg)
    g = SemiImplicitSolver(mesh, HLLCSolver(eos), SOLVERS[kind](), eos, None, cfg)
    pg, pc = np.zeros(mesh.totalCells()), np.zeros(mesh.totalCells())
    ig = SOLVERS[kind](g).solve(mesh, rho, rhoc2, rhs, pg, dt, tol, 2000)
    g.close()
    cpu = oracle_c.CpuSolver(mesh, cfg, 2, eos, "c")
    ic = (cpu.pcg if kind == "PCG" else cpu.mgpcg)(rho, rhoc2, rhs, pc, dt, tol, 2000)
    assert 0 < ig < 2000 and abs(ig - ic) <= max(2, ic // 10), (ig, ic)
    ref = mesh.interior(pc)
    assert np.isfinite(ref).all()
    assert np.abs(mesh.interior(pg) - ref).max() <= 1e3 * tol * np.abs(ref).max()


def _residual(mesh, rho, rhoc2, rhs, p, dt):
    """||rhs - (1 + c L) p|| / ||rhs|| over the interior, row by row in FP64: the face
    coefficients 1 / (max(rho_face, 1e-14) distance h) of the solved system, 0 at walls."""
    I = mesh.interior
    r, q, c = I(rho), I(p), I(rhoc2) * dt * dt
    acc = q - I(rhs)
    for axis, width in enumerate((mesh.dz, mesh.dy, mesh.dx)):
        n = r.shape[axis]
        if n == 1:
            continue
        wrap = mesh.periods[2 - axis]
        h = np.array([width(m) for m in range(n)]).reshape([-1 if a == axis else 1 for a in range(3)])
        rn, qn, hn = (np.roll(v, -1, axis) for v in (r, q, np.broadcast_to(h, r.shape)))
        face = 1.0 / (np.maximum(0.5 * (r + rn), 1e-14) * 0.5 * (h + hn))   # high face of each cell
        if not wrap:
            face[tuple(-1 if a == axis else slice(None) for a in range(3))] = 0.0
        flux = face * (qn - q)
        acc = acc - c / h * (flux - np.roll(flux, 1, axis))
    return np.linalg.norm(acc) / np.linalg.norm(I(rhs))


@pytest.mark.parametrize("kind", ["PCG", "MGPCG"])
@pytest.mark.parametrize("shape,periods", [SHAPES[0], SHAPES[1], SHAPES[2], SHAPES[4]])
def test_pcg_residual_under_the_floor(gpu, shape, periods, kind):
    """The answer's own residual under the rows of the system with floored densities is
    within the tolerance that the solve stopped at (1 % for the recurrence's rounding;
    without the floor the 1000:1 system's plateau lies above the tolerance)."""
    cfg, mesh, rho, rhoc2, rhs, dt = _system(shape, periods, True)
    eos = IdealGasEOS(1.4, 1.0, cfg)
    g = SemiImplicitSolver(mesh, HLLCSolver(eos), SOLVERS[kind](), eos, None, cfg)
    p = np.zeros(mesh.totalCells())
    its = SOLVERS[kind](g).solve(mesh, rho, rhoc2, rhs, p, dt, 1e-7, 2000)
    g.close()
    res = _residual(mesh, rho, rhoc2, rhs, p, dt)
    assert 0 < its < 2000 and res <= 1.01e-7, (its, res)
