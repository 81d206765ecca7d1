"""The sweep kernels at the sizes where their tilings can go wrong: lines of
one node, lines that end in a partial segment, lines one node longer than a
tile holds, more lines than a block and fewer, against the CPU oracle on the
same inputs (exact arithmetic: bit for bit where no pow() is involved)."""
import os
import sys

import numpy as np
import pytest

from conftest import ROOT

sys.path.insert(0, os.path.join(ROOT, "cases"))
import make_cases as mc  # noqa: E402

pytestmark = pytest.mark.gpu

INIT = ("1+0.2*sin(6*x)*cos(4*y)", "0.3", "0.2*cos(3*x+5*z)", "0.1*sin(7*y)", "1")
OPEN = [mc.inflow(1.1, 0.4, 0.1, 0, 1.2)] + [mc.OUTFLOW] * 5
RING = [mc.PERIODIC] * 6
WALLS = [mc.slip(), mc.noslip(), mc.noslip(0.0033), mc.slip(0.0036), mc.slip(), mc.noslip()]


def write_case(tmp_path, m, bcs, numerical=mc.DEFAULT_NUM, mu=0.0):
    d = tmp_path / "case"
    d.mkdir()
    h = 0.02
    length = tuple(h * max(v, 1) for v in m)
    jump = mc.box((-9, -9, -9), (0.4 * length[0], 0.6 * length[1], 9), (0.6, 0.1, -0.2, 0.05, 0.5))
    (d / "artracfd.case").write_text(mc.case_text(((0, 0, 0), length, m), (0, 1e9, 0.6, 0, 1, 0), numerical,
                                                  (0, mu, 0, (0, 0, 0)), mc.REF1, INIT, bcs, [jump]))
    (d / "artracfd.geo").write_text(mc.geo_text())
    return str(d)


def against_oracle(oracle_mod, directory, steps, exact, **options):
    """(device interior, oracle interior, fused axes) after `steps` steps."""
    from artracfd_amd import Case, Solver
    case = Case(directory)
    oracle_mod.treat_boundary(case, 0)
    done, dts = oracle_mod.march(case, steps)
    ref = case.interior(case.field()).copy()
    case.close()
    case = Case(directory)
    solver = Solver(case, exact=exact, **options)
    axes = solver.fused_axes()
    got, gdts = solver.march(steps)
    U = case.interior(solver.field()).copy()
    solver.close()
    case.close()
    assert got == done == steps
    np.testing.assert_allclose(gdts, dts, rtol=1e-13)
    return U, ref, axes


# interior nodes per axis are m - 1 (open faces) or m + 1 (periodic)
STAGES = [((2, 3, 4), OPEN, 0.0), ((258, 4, 3), OPEN, 0.0), ((3, 130, 5), OPEN, 0.0), ((4, 3, 66), RING, 0.0),
          ((53, 29, 7), RING, 0.02), ((2, 33, 2), RING, 0.02), ((131, 3, 20), OPEN, 0.02), ((11, 37, 16), WALLS, 0.0)]


@pytest.mark.parametrize("m, bcs, mu", STAGES)
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("numerical", [(1, 1, 0, 0, 0, 0, 1), (0, 0, 1, 1, 1, 0, 1)])
def test_stage_sweeps_at_the_edges_of_their_tiles(tmp_path, oracle_mod, m, bcs, mu, exact, numerical):
    """Stage-by-stage sweeps (split WENO5-RK3 and unsplit Roe WENO3-RK2): the
    fast arithmetic and the viscous flux's pow() stay at rounding level,
    1e-13 of the largest value of a group after two steps."""
    print(m, mu, exact, numerical, flush=True)
    U, ref, _ = against_oracle(oracle_mod, write_case(tmp_path, m, bcs, numerical, mu), 2, exact, fused=False)
    if exact and mu == 0.0:
        assert np.array_equal(U, ref)
    for c in (slice(0, 1), slice(1, 4), slice(4, 5)):
        assert np.abs(U[c] - ref[c]).max() <= 1e-13 * np.abs(ref[c]).max()
