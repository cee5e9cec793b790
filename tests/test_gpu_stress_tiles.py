"""Face stresses (visc_kernel) at the edges of its tiles: 64 columns x 8 rows
per block (256 columns in 1D) and 8 planes of z, with meshes one cell short of,
at and one cell past them, against the oracle.

Bars: single phase 1e-12 relative Linf (the viscous tests' bar).  Water/air
1e-9: the pressure is the difference of energies ~3e9 in FP64 (6e-7 Pa of
rounding against 1e5 Pa, 6e-12 relative) and each of the 2 steps' 3 stages
carries a few such roundings into the momenta."""
import pytest

from semiimplicitfv_amd import BoundaryCondition as BC, ExplicitSolver, HLLCSolver
from tests.golden import problems
from tests.helpers import rel_errs

pytestmark = pytest.mark.gpu

BCS = [BC.NoSlipWall, BC.SlipWall, BC.SlipWall, BC.NoSlipWall, BC.Outflow, BC.NoSlipWall]
SIZES = [(255,), (257,), (63, 9), (64, 8), (65, 7), (130, 17), (65, 9, 7), (63, 8, 9), (66, 17, 8)]


def _run(po, cfg, mesh, st, eos, steps=2):
    g = ExplicitSolver(mesh, HLLCSolver(eos), eos, None, cfg)
    c = po.CpuSolver(mesh, cfg, 2, eos, "c")
    sc = st.copy()
    g.upload(st)
    for k in range(steps):
        cfg.step = k
        g.step_resident(cfg)
        c.explicit_step(sc, cfg)
    g.download(st)
    g.close()
    return max(rel_errs(mesh.interior(st.field(f)), mesh.interior(sc.field(f)))[1] for f in st.field_ids()
               if abs(mesh.interior(sc.field(f))).max() > 0.0)


@pytest.mark.parametrize("n", SIZES)
def test_viscous_tiles(gpu, oracle_c, n):
    cfg, mesh, st, eos = problems.make_case(len(n), n, bcs=BCS, periods=(0, 0, 0) if len(n) < 3 else (1, 0, 0), seed=51,
                                            nonuniform=True, cfl=0.4)
    cfg.viscousParams.mu = 1e-2
    assert _run(oracle_c, cfg, mesh, st, eos) <= 1e-12


@pytest.mark.parametrize("n", [s for s in SIZES if len(s) > 1])
def test_capillary_tiles(gpu, oracle_c, n):
    cfg, mesh, st, eos = problems.make_two_phase_case(len(n), n, bcs=BCS, seed=53, p_jump=False,
                                                      nonuniform=True)
    cfg.surfaceTensionParams.sigma = 1e3
    cfg.viscousParams.phaseMu = [5.0, 0.5]
    assert _run(oracle_c, cfg, mesh, st, eos) <= 1e-9
