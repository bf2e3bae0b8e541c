"""Least-squares gradients whose weights are formed in the kernel from the centroids, against the
oracle's stored weights: all boundary kinds, rows whose length leaves 0, 1, 2 or 3 entries for the
last batch, one to five fields in a pass. Both forms of the row on every mesh."""
import numpy as np
import pytest

import oracle
from dopamine_amd import cases
from dopamine_amd.solver import FVSolver
from helpers import rel_l2, run_case
from hostcheck import HostSolver, lib

CASES = {
    "tgv_skew": lambda: cases.regression_cases()["tgv_skew"],    # periodic all round
    "hydrowall": lambda: cases.regression_cases()["hydrowall"],  # walls
    "pdrop": lambda: cases.regression_cases()["pdrop"],          # inlet and outlet
    "channel": lambda: cases.small_channel(16, 12, 8),           # velocity and SGS viscosity
    "thin": lambda: cases.small_channel(5, 7, 2),                # two cells across a periodic direction
    "tets": lambda: cases.cavity_tets(5),                        # rows of 12 to 32 entries
    "rb": lambda: cases.rayleigh_benard(12, 12, 8),              # temperature
    "most": lambda: cases.most_channel(12, 8, 6),                # temperature, list of wall cells
    "full": lambda: cases.full_stack(16, 16, 8, n_obstacles=3, seed=5),  # temperature and two scalars
}


def case_of(name):
    case = CASES[name]()
    case.params.p_tol = 1e-12
    return case


def compare(make, name):
    case = case_of(name)
    mesh = case.make_mesh()
    print(f"least-squares rows {name}: {mesh.n_cells} cells", flush=True)
    s, o = make(mesh, case.params), oracle.Solver(mesh, case.params)
    for q in (s, o):
        run_case(q, case, mesh, nsteps=2, stats_every=2)
    # the bar of the plain-FP64 fields; the weights themselves agree to 1e-12 of the row's largest,
    # so one gradient of a field of order 1 to about 32 x 1e-12 of its largest term
    assert rel_l2(o.U, s.U) < 1e-10
    return s


@pytest.mark.parametrize("form", ["0", "1"])
@pytest.mark.parametrize("name", CASES)
def test_fields_match_the_oracle(name, form, monkeypatch):
    monkeypatch.setenv("DOPAMINE_LS_GEOMETRY", form)
    s = compare(HostSolver, name)
    assert lib().hc_ls_geometry(s.h) == int(form)


@pytest.mark.parametrize("name,form", [("channel", 1), ("full", 1), ("tets", 0)])
def test_form_follows_the_numbering(name, form, monkeypatch):
    monkeypatch.delenv("DOPAMINE_LS_GEOMETRY", raising=False)
    case = case_of(name)
    assert lib().hc_ls_geometry(HostSolver(case.make_mesh(), case.params).h) == form


def test_other_weights_are_taken_as_they_are(monkeypatch):
    monkeypatch.setenv("DOPAMINE_LS_GEOMETRY", "1")
    case = case_of("channel")
    mesh = case.make_mesh()
    mesh.ls_weight = mesh.ls_weight * (1.0 + 1e-9)
    assert lib().hc_ls_geometry(HostSolver(mesh, case.params).h) == 0


def test_one_cell_across_a_periodic_direction(monkeypatch):
    """A cell that is its own periodic neighbour."""
    monkeypatch.setenv("DOPAMINE_LS_GEOMETRY", "1")
    case = cases.small_channel(6, 6, 1)
    mesh = case.make_mesh()
    s, o = HostSolver(mesh, case.params), oracle.Solver(mesh, case.params)
    for q in (s, o):
        run_case(q, case, mesh, nsteps=1, stats_every=1)
    assert rel_l2(o.U, s.U) < 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("name", CASES)
def test_gpu_fields_match_the_oracle(name, monkeypatch):
    monkeypatch.setenv("DOPAMINE_LS_GEOMETRY", "1")
    compare(FVSolver, name)


def compare_scalars(make, n_scalars):
    """Three and four scalars beside the velocity and the temperature."""
    case = cases.full_stack(12, 12, 8, n_obstacles=2, seed=7)
    case.params.p_tol = 1e-12
    case.params.n_scalars = n_scalars
    case.params.scalar_diffusivity = (0.1, 0.2, 0.3, 0.4)
    mesh = case.make_mesh()
    print(f"least-squares rows, {n_scalars} scalars", flush=True)
    s, o = make(mesh, case.params), oracle.Solver(mesh, case.params)
    x = mesh.cell_centroid / 100.0
    for q in (s, o):
        run_case(q, case, mesh, nsteps=1, stats_every=1)
        for k in range(n_scalars):
            q.set_scalar(k, np.sin((k + 1) * x[:, 0]) + x[:, 2])
        q.advance()
    assert max(rel_l2(o.scalar(k), s.scalar(k)) for k in range(n_scalars)) < 1e-10
    assert rel_l2(o.U, s.U) < 1e-10


@pytest.mark.parametrize("n_scalars", [3, 4])
def test_more_scalars(n_scalars, monkeypatch):
    monkeypatch.setenv("DOPAMINE_LS_GEOMETRY", "1")
    compare_scalars(HostSolver, n_scalars)


@pytest.mark.gpu
@pytest.mark.parametrize("n_scalars", [3, 4])
def test_gpu_more_scalars(n_scalars, monkeypatch):
    monkeypatch.setenv("DOPAMINE_LS_GEOMETRY", "1")
    compare_scalars(FVSolver, n_scalars)
