"""The sweep kernels at the sizes where their tilings can go wrong: lines of
one node, lines that end in a partial segment, lines one node longer than a
tile holds, more lines than a block and fewer, against the CPU oracle on the
same inputs (exact arithmetic: bit for bit where no pow() is involved)."""
import os
import sys

import numpy as np
import pytest

import mlp_oracle as M
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


def test_viscous_face_between_nodes_without_pressure(tmp_path):
    """Two neighbours along z with E = rho w^2 / 2 exactly: their temperature
    and Sutherland's viscosity at their face are zero in both arithmetics."""
    from artracfd_amd import Case, Solver
    directory = write_case(tmp_path, (7, 7, 7), RING, mu=0.02)
    out = []
    for exact in (True, False):
        case = Case(directory)
        solver = Solver(case, exact=exact)
        U = solver.field()
        U[:, 5, 6, 6] = [1.0, 0.0, 0.0, 0.5, 0.125]
        U[:, 6, 6, 6] = [1.0, 0.0, 0.0, 0.25, 0.03125]
        solver.set_field(0, U)
        print(exact, flush=True)
        solver.evolve(1e-6)
        out.append(case.interior(solver.field()).copy())
        solver.close()
        case.close()
    assert np.isfinite(out[0]).all()
    for c in (slice(0, 1), slice(1, 4), slice(4, 5)):
        assert np.abs(out[1][c] - out[0][c]).max() <= 1e-13 * np.abs(out[0][c]).max()


MIXED = [mc.inflow(1.1, 0.4, 0.1, 0, 1.2), mc.noslip(), mc.slip(), mc.OUTFLOW, mc.noslip(0.0033), mc.slip(0.0036)]
# (nodes, boundaries, the axes that run as lines): lines of one node to one
# past the two-node threads' first, the longest line and one longer, several
# lines to a block with a rest, a wavefront's and a block's faces more or less
# by one
LINES = [((2, 3, 4), OPEN, "xyz"), ((4, 3, 3), RING, "xyz"), ((64, 63, 5), OPEN, "xyz"), ((4, 128, 7), RING, "xyz"),
         ((256, 3, 5), OPEN, "xyz"), ((257, 5, 3), OPEN, "xyz"), ((3, 512, 3), OPEN, "xyz"), ((3, 3, 513), OPEN, "xyz"),
         ((3, 511, 3), RING, "xyz"), ((3, 3, 514), OPEN, "xy"),
         ((11, 37, 16), WALLS, "xyz"), ((4, 258, 4), WALLS, "xyz"), ((21, 4, 66), MIXED, "xyz"),
         ((2, 7, 2), WALLS, "y")]                # (a wall needs as many interior nodes as ghosts)


@pytest.mark.parametrize("m, bcs, expected", LINES)
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("numerical", [(1, 1, 0, 0, 0, 0, 1), (0, 0, 0, 1, 1, 0, 1)])
def test_lines_at_the_edges_of_their_blocks(tmp_path, oracle_mod, m, bcs, expected, exact, numerical):
    """Whole operators on lines in local memory against the oracle: bit for
    bit in exact arithmetic, rounding level (1e-13 of the largest value of a
    group after two steps) in the fast one, with any kind of boundary at the
    lines' ends."""
    print(m, exact, numerical, flush=True)
    U, ref, axes = against_oracle(oracle_mod, write_case(tmp_path, m, bcs, numerical), 2, exact)
    print("axes", axes)
    assert "".join("xyz"[a] for a in axes) == expected
    if exact:
        assert np.array_equal(U, ref)
    for c in (slice(0, 1), slice(1, 4), slice(4, 5)):
        assert np.abs(U[c] - ref[c]).max() <= 1e-13 * np.abs(ref[c]).max()


@pytest.mark.parametrize("bcs", [OPEN, RING, MIXED])
def test_a_step_on_lines_starts_from_the_ghosts_of_its_input(tmp_path, bcs):
    """One step on a caller's field with ghosts of its own: the first operator
    reads them as they are, on lines as stage by stage."""
    from artracfd_amd import Case, Solver
    directory = write_case(tmp_path, (9, 70, 6), bcs)
    out = []
    for fused in (True, False):
        case = Case(directory)
        solver = Solver(case, exact=True, fused=fused)
        U = solver.field()
        solver.set_field(0, U * (1.0 + 1e-3 * np.cos(np.arange(U.size)).reshape(U.shape)))
        print(bcs[0], fused, flush=True)
        solver.evolve(1e-4)
        out.append(case.interior(solver.field()).copy())
        solver.close()
        case.close()
    assert np.array_equal(out[0], out[1])


IN_LOW, IN_HIGH = mc.inflow(1.1, 0.1, 0.2, 0.4, 1.2), mc.inflow(0.9, -0.2, 0.1, -0.3, 0.8)
INFLOWS = {"low": [mc.OUTFLOW] * 4 + [IN_LOW, mc.OUTFLOW], "high": [mc.OUTFLOW] * 4 + [mc.OUTFLOW, IN_HIGH],
           "both": [mc.OUTFLOW, IN_HIGH, IN_LOW, IN_HIGH, IN_LOW, IN_HIGH],
           "wall": [IN_LOW, mc.slip(), IN_LOW, mc.noslip(), IN_LOW, mc.noslip(0.0033)],
           "x": [IN_LOW, mc.OUTFLOW] + [mc.OUTFLOW] * 4, "y": [mc.OUTFLOW] * 2 + [mc.OUTFLOW, IN_HIGH] + [mc.OUTFLOW] * 2}


def with_ghosts_of_its_own(solver, scale=1e-3):
    """Every node's state changed, the ghosts' too: they no longer are what a
    boundary fill makes of the interior."""
    U = solver.field()
    solver.set_field(0, U * (1.0 + scale * np.cos(np.arange(U.size)).reshape(U.shape)))


def run_once(directory, steps, start=with_ghosts_of_its_own, params=None, threshold=0.0, gate=0.0, **options):
    """Interior after evolve() (steps 0) or a march, from the field `start` makes."""
    from artracfd_amd import Case, Solver
    case = Case(directory)
    solver = Solver(case, **options)
    if params is not None:
        solver.set_indicator(params, threshold, smooth_variation=gate)
    start(solver)
    if steps:
        assert solver.march(steps)[0] == steps
    else:
        solver.evolve(1e-4)
    U = case.interior(solver.field()).copy()
    solver.close()
    case.close()
    return U


# the first operator runs along z in three dimensions, along y with z
# collapsed, along the one axis of a tube (both operators in one launch)
@pytest.mark.parametrize("m, kind", [((6, 5, 70), "low"), ((6, 5, 70), "high"), ((6, 5, 70), "both"),
                                     ((5, 6, 40), "wall"), ((4, 4, 300), "both"), ((40, 30, 1), "y"),
                                     ((40, 30, 1), "both"), ((70, 1, 1), "x"), ((1, 1, 70), "low"),
                                     ((1, 70, 1), "y")])
@pytest.mark.parametrize("steps", [0, 3])
@pytest.mark.parametrize("numerical", [(1, 1, 0, 0, 0, 0, 1), (0, 0, 0, 1, 1, 0, 1)])
def test_prescribed_states_are_back_after_the_first_stage(tmp_path, m, kind, steps, numerical):
    """A call that starts from a caller's own ghosts reads them in its first
    stage only: from then on an inflow end holds its prescribed state, on
    lines as stage by stage."""
    directory = write_case(tmp_path, m, INFLOWS[kind], numerical)
    print(m, kind, steps, flush=True)
    fused = run_once(directory, steps, exact=True)
    assert np.array_equal(fused, run_once(directory, steps, exact=True, fused=False))


@pytest.mark.parametrize("m, kind", [((4, 3, 70), "both"), ((3, 3, 300), "low"), ((70, 1, 1), "x")])
@pytest.mark.parametrize("steps", [0, 3])
def test_prescribed_states_on_routed_lines(tmp_path, m, kind, steps):
    """The same with the indicator: every face on the full flux is the plain
    solver bit for bit (lines deferred by the lean pass and, beyond 256
    nodes, lines that never take it)."""
    directory = write_case(tmp_path, m, INFLOWS[kind])
    print(m, kind, steps, flush=True)
    plain = run_once(directory, steps)
    assert np.array_equal(plain, run_once(directory, steps, params=M.init_params(3), threshold=-1e30))


def test_prescribed_states_on_lean_lines(tmp_path):
    """A smooth line stays in the lean pass; the same line with a jump at its
    far end is deferred and routed.  Near the inflow both take the linear flux
    and agree bit for bit, from ghosts of their own."""
    directory = write_case(tmp_path, (1, 1, 200), INFLOWS["low"])
    out = []
    for jump in (0.0, 0.5):
        def start(solver):
            U = np.ones_like(solver.field()) * np.array([1.1, 0.11, 0.22, 0.44, 3.2])[:, None, None, None]
            U *= 1.0 + 2e-4 * np.cos(np.arange(U.size)).reshape(U.shape)
            U[:, 160:] *= 1.0 + jump
            solver.set_field(0, U)
        print("jump", jump, flush=True)
        out.append(run_once(directory, 0, start, params=M.init_params(3), threshold=-1e30, gate=1e-2)[:, :60])
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("routed", [False, True])
def test_batched_lines_start_from_the_ghosts_of_their_input(tmp_path, routed):
    """A batch started from ghosts of its own gives what its cases give alone."""
    from artracfd_amd import Case, Solver
    from artracfd_amd.batch import Batch
    dirs = []
    for q, (m, kind) in enumerate([((5, 4, 70), "both"), ((12, 11, 40), "low"), ((6, 5, 256), "high")]):
        (tmp_path / str(q)).mkdir()
        dirs.append(write_case(tmp_path / str(q), m, INFLOWS[kind]))
    cases = [Case(d) for d in dirs]
    solvers = [Solver(c) for c in cases]
    for s in solvers:
        with_ghosts_of_its_own(s)
    print("batch", routed, flush=True)
    b = Batch(solvers)
    if routed:
        b.set_indicator(M.init_params(3), -1e30)
    b.march(3)
    got = [c.interior(s.field()).copy() for c, s in zip(cases, solvers)]
    b.close()
    for s, c in zip(solvers, cases):
        s.close()
        c.close()
    alone = dict(params=M.init_params(3), threshold=-1e30, gate=1e-3) if routed else {}
    for q, d in enumerate(dirs):
        assert np.array_equal(got[q], run_once(d, 3, **alone)), q


def test_batched_lines_at_the_edges_of_their_blocks(tmp_path):
    """Lines of 2 to 257 faces packed into one batch give what
    the cases give alone, bit for bit."""
    from artracfd_amd import Case, Solver
    from artracfd_amd.batch import Batch
    dirs = []
    for q, m in enumerate([(2, 3, 4), (63, 5, 3), (255, 4, 3), (4, 257, 6)]):
        (tmp_path / str(q)).mkdir()
        dirs.append(write_case(tmp_path / str(q), m, OPEN if q % 2 else RING))
    alone = []
    for d in dirs:
        case = Case(d)
        solver = Solver(case)
        solver.march(3)
        alone.append(case.interior(solver.field()).copy())
        solver.close()
        case.close()
    cases = [Case(d) for d in dirs]
    solvers = [Solver(c) for c in cases]
    print("batch", flush=True)
    b = Batch(solvers)
    b.march(3)
    for q, (c, s) in enumerate(zip(cases, solvers)):
        assert np.array_equal(c.interior(s.field()), alone[q]), q
    b.close()
    for s, c in zip(solvers, cases):
        s.close()
        c.close()


@pytest.mark.parametrize("m, r, steps", [(64, 0.41, 3), (24, 0.2, 4)])
def test_flags_of_a_moving_body_reach_the_host(tmp_path, m, r, steps):
    """The host's flags after half-steps that change thousands of nodes (more
    than one copy of the changes holds) and few: the domain field is the
    sphere at its last position, interfacial layer 1 its nodes with a fluid
    neighbour, ghosts exactly the body's interfacial nodes."""
    from artracfd_amd import Case, Solver
    d = tmp_path / "case"
    d.mkdir()
    (d / "artracfd.case").write_text(mc.case_text(((-0.5, -0.5, -0.5), (0.5, 0.5, 0.5), (m, m, m)),
                                                  (0, 1e9, 0.6, 0, 1, 0), (1, 1, 0, 0, 0, 1, 1), mc.INVISCID, mc.REF1,
                                                  ("1", "0", "0", "0", "1"), [mc.OUTFLOW] * 6))
    (d / "artracfd.geo").write_text(mc.moving_geo_text(spheres=[
        dict(O=(-0.02, 0.01, 0.0), r=r, V=(3.0, 1.0, 0.5), rho=50.0, mid=2)]))
    case = Case(str(d))
    solver = Solver(case)
    before = case.interior(case.flags()).copy()
    print(m, r, flush=True)
    done, _ = solver.march(steps)
    flags, O = case.interior(case.flags()), case.bodies()[0, :3]
    assert done == steps and np.isfinite(case.interior(solver.field())).all()
    x = [-0.5 + (np.arange(*case.pin[s]) - (case.n[s] - m - 1) // 2) / m - O[s] for s in range(3)]
    d2 = x[2][:, None, None] ** 2 + x[1][None, :, None] ** 2 + x[0][None, None, :] ** 2
    inside = flags[0] == 1
    assert (inside == (d2 <= r * r))[np.abs(d2 - r * r) > 1e-12].all()
    near = np.zeros_like(inside)
    for axis in range(3):
        for shift in (1, -1):
            near |= np.roll(~inside, shift, axis)
    assert np.array_equal(flags[2] == 1, inside & near)
    assert np.array_equal(flags[3] == 1, inside & near)
    if m == 64:
        assert (flags != before).any(axis=0).sum() > 1024
    solver.close()
    case.close()


def test_boxes_of_moving_bodies_are_those_of_their_nodes(tmp_path):
    """The boxes that bound the next classification, from the device, after
    every step: a body that crosses the grid, one that leaves it, one at rest
    (tests/scope_device.c)."""
    import subprocess

    from artracfd_amd import library
    d = tmp_path / "case"
    d.mkdir()
    m = 32
    (d / "artracfd.case").write_text(mc.case_text(((-0.5, -0.5, -0.5), (0.5, 0.5, 0.5), (m, m, m)),
                                                  (0, 1e9, 0.6, 0, 1, 0), (1, 1, 0, 0, 0, 1, 1), mc.INVISCID, mc.REF1,
                                                  ("1", "0", "0", "0", "1"), [mc.OUTFLOW] * 6))
    (d / "artracfd.geo").write_text(mc.moving_geo_text(spheres=[
        dict(O=(-0.3, -0.2, 0.0), r=0.11, V=(2.0, 1.0, 0.5), rho=50.0, mid=2),
        dict(O=(0.38, 0.3, 0.3), r=0.1, V=(4.0, 1.0, 1.0), rho=50.0, mid=2),
        dict(O=(-0.3, 0.3, -0.3), r=0.12, rho="1e37", mid=2)]))
    lib = library()._name
    exe = str(tmp_path / "scope_device")
    subprocess.run(["gcc", "-O1", "-std=c11", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "artracfd_amd", "csrc", "host"),
                    os.path.join(ROOT, "tests", "scope_device.c"), "-o", exe, lib, "-Wl,-rpath," + os.path.dirname(lib),
                    "-lm"], check=True)
    print("scope_device", flush=True)
    out = subprocess.run([exe, str(d), "24"], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.split() == ["ok", "24", "1"], out.stdout
