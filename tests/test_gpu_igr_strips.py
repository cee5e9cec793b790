"""2D strip streaming of the IGR sweeps at the edges of its forms: the fewest rows
it takes, one strip of one lane's or of 64 columns, a last strip of one column,
strips that all end at walls, periods with and without idle rows, sweep counts of
one and two (edge values of both parities), and wide meshes whose record slots
repeat within a period.  Against the oracle's lexicographic sweeps, to the bar of
rel L1 and Linf <= 1e-12 that the solver's other strip tests have."""
import pytest

from semiimplicitfv_amd import ExplicitSolver, LFSolver
from tests.helpers import rel_errs
from tests.test_gpu_igr import _wavefront_case

pytestmark = pytest.mark.gpu

# mesh, wrapping axes, sweeps at the first step, sweeps afterwards, steps
STRIPS = {
    "fewest_rows_per_xy": ((128, 152), (1, 1, 0), 6, 3, 2),
    "one_full_strip_walls": ((64, 157), (0, 0, 0), 5, 1, 3),
    "one_full_strip_per_x": ((64, 153), (1, 0, 0), 2, 1, 3),
    "eight_columns_per_xy": ((8, 191), (1, 1, 0), 5, 2, 2),
    "last_strip_one_column_walls": ((129, 160), (0, 1, 0), 7, 2, 2),
    "period_without_idle_rows": ((70, 400), (1, 1, 0), 6, 3, 2),
    "slots_repeat_in_a_period": ((6720, 152), (1, 1, 0), 3, 2, 2),
    "slots_of_the_rows_alone": ((704, 200), (1, 1, 0), 3, 2, 2),
    "slots_of_some_idle_rows_walls_y": ((400, 190), (1, 0, 0), 3, 2, 2),
}


@pytest.mark.parametrize("key", list(STRIPS))
def test_igr_strip_forms(gpu, oracle_c, key):
    n, periods, warm, iters, nsteps = STRIPS[key]
    cfg, mesh, st, eos = _wavefront_case(2, n, periods, warm, iters, seed=31)
    sg, sc = st.copy(), st.copy()
    gpu_s = ExplicitSolver(mesh, LFSolver(eos), eos, None, cfg)
    cpu = oracle_c.CpuSolver(mesh, cfg, 0, eos, "c")
    gpu_s.upload(sg)
    for k in range(nsteps):
        cfg.step = k
        dg = gpu_s.step_resident(cfg)
        dc = cpu.explicit_step(sc, cfg)
        assert abs(dg - dc) <= 1e-13 * dc
    gpu_s.download(sg)
    gpu_s.close()
    for fid in sc.field_ids():
        l1, li = rel_errs(mesh.interior(sg.field(fid)), mesh.interior(sc.field(fid)))
        assert l1 <= 1e-12 and li <= 1e-12, (fid, l1, li)
