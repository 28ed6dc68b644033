"""Explicit Runge-Kutta stages (a_ss = 0) in the explicit HDG modes, which run without a condensation, against the
general element kernel on the same problem (that one is pinned to the oracle in test_runge_kutta_gpu.py): every order,
the first and a later stage, both explicit modes, with and without the fused scatter; and the neighbouring schemes
that keep the full condensation.

Bound: both sides are FP64 sums of a few hundred terms and one mass solve; 1e-11 of the largest value is the bar that
the general kernel itself is held to against the oracle."""
import numpy as np
import pytest

import hyperfox_amd as hf
import hyperfox_amd.problems as pr
from hdg_helpers import rel
from test_gpu_parity import run_gpu, small_workload
from test_runge_kutta_gpu import random_fields, set_fields

pytestmark = pytest.mark.gpu


def assembled(w, kernel, fused, table, stage, mode, seed=31):
    prob, _ = run_gpu(w)
    prob.set_kernel(kernel)
    prob.set_fused_scatter(fused)
    set_fields(prob, *random_fields(w, seed))
    prob.set_solver_type(mode)
    prob.set_time_scheme(hf.TS_RK, 0.03)
    prob.set_butcher(table)
    prob.rk_start_step()
    for s in range(stage):
        prob.assemble()
        prob.solve(pc=hf.PC_BJACOBI, rtol=1e-13, maxits=50)
        prob.rk_compute_stage()
    prob.assemble()
    return prob.condensed(), prob.trace_csr()


@pytest.mark.parametrize('fused', [True, False])
@pytest.mark.parametrize('mode', [hf.HDG_WEXPLICIT, hf.HDG_SEXPLICIT])
@pytest.mark.parametrize('table,stage', [('FEuler', 0), ('RK4', 2)])
@pytest.mark.parametrize('kind', [0, 2])
@pytest.mark.parametrize('dim,p', [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3)])
def test_stage_matches_the_general_kernel(dim, p, kind, table, stage, mode, fused):
    print('explicit stage', dim, p, kind, table, stage, mode, fused, flush=True)
    w = small_workload(dim, p, kind)
    g, (_, _, vg, rg) = assembled(w, 1, False, table, stage, mode)
    x, (_, _, vx, rx) = assembled(w, 0, fused, table, stage, mode)
    assert not x['U'].any() and not g['U'].any()
    for k in ('S', 'S0', 'Q', 'U0', 'Q0'):
        assert rel(x[k], g[k]) < 1e-11, k
    assert rel(vx, vg) < 1e-11 and rel(rx, rg) < 1e-11


@pytest.mark.parametrize('table,mode', [('ALX2', hf.HDG_SEXPLICIT), ('RK4', hf.HDG_IMPLICIT)])
def test_other_stages_keep_the_condensation(table, mode):
    """A stage with a_ss != 0, and an explicit stage in the implicit HDG mode (S couples the faces)."""
    w = small_workload(3, 2, 2)
    g, (_, _, vg, rg) = assembled(w, 1, False, table, 0, mode)
    x, (_, _, vx, rx) = assembled(w, 0, True, table, 0, mode)
    for k in ('S', 'S0', 'U', 'Q', 'U0', 'Q0'):
        assert rel(x[k], g[k]) < 1e-11 or not g[k].any(), k
    assert rel(vx, vg) < 1e-11 and rel(rx, rg) < 1e-11


def test_explicit_stage_on_more_cells_than_wavefronts():
    w = pr.diffusion_source_2d(70, 1)  # 9,800 cells: several cells per wavefront
    g, (_, _, vg, rg) = assembled(w, 1, False, 'SSPRK3', 1, hf.HDG_SEXPLICIT)
    x, (_, _, vx, rx) = assembled(w, 0, True, 'SSPRK3', 1, hf.HDG_SEXPLICIT)
    for k in ('S', 'S0', 'Q', 'U0', 'Q0'):
        assert rel(x[k], g[k]) < 1e-11, k
    assert rel(vx, vg) < 1e-11 and rel(rx, rg) < 1e-11
