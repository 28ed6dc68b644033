"""The multi-component cell kernel with more cells than workgroups: each workgroup takes several cells through the same
LDS, where the blocks of a later phase lie over the arrays of an earlier one. Against the oracle, at the bound that the
blocks of single cells are held to (test_burgers_gpu.py); the small state keeps every cell's system diffusive, so that
its condition does not eat into that bound."""
import pytest

from test_burgers_gpu import gpu_problem, oracle_problem, rel, workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dim,p,n', [(2, 1, 26), (2, 3, 23), (3, 1, 6)])
def test_several_cells_per_workgroup(dim, p, n):
    print('cells per workgroup', dim, p, n, flush=True)
    mesh, fields, state = workload(dim, p, n=n)
    state['buffer'] *= 0.1
    state['trace'] *= 0.1
    prob = gpu_problem(dim, p, mesh, fields, state)
    prob.assemble()
    got = prob.condensed()
    orc = oracle_problem(dim, p, mesh, fields)
    orc.assemble(state['buffer'].reshape(mesh.n_cells, -1), state['trace'])
    for name, g, o in zip(('S', 'S0', 'U', 'Q', 'U0', 'Q0'), got, (orc.S, orc.S0, orc.U, orc.Q, orc.U0, orc.Q0)):
        assert rel(g, o) < 1e-10, name
