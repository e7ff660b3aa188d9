"""The step's alternative paths give what the path they stand in for gives.

A solve's arithmetic does not depend on the path that its handle takes, so the bar is equality of
every bit: small solves that fill their own ghosts in a sequence of steps against the same steps one
at a time, steps from flux tables against weights formed in the step, general-step tracers launched
together against each alone, and read-outs through pinned staging against a plain copy.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device visible")


def _steady(ntr):
    from cubedsphere.cases import random_solid_body
    return random_solid_body(np.random.default_rng(ntr), ntr)


def _unsteady(ntr):
    from cubedsphere.cases import Case, workload
    c = workload("nl10_deformation")
    return Case(c.tracers[:ntr], c.wind)


def _run(N, case, parts, graph=0, dtype="f64", **kw):
    from cubedsphere.solver import Advection
    sol = Advection(N, case, 0.2 / N, dtype=dtype, device="cuda:0", max_steps=sum(parts), **kw).init_vars_adv()
    if graph:
        sol.use_graph(graph)
    for n in parts:
        sol.step(n)
    out = sol.full_state(), sol.state(), [sol.mass(t) for t in range(case.ntr)]
    sol.close()
    return out


def _same(a, b):
    assert np.isfinite(a[1]).all()
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


# N: one segment of rows, a last segment of one and of two rows, several strips; tile 1 has its own split
@pytest.mark.parametrize("N,tile", [(12, 0), (17, 0), (18, 0), (33, 0), (50, 0), (65, 0), (33, 1)])
@pytest.mark.parametrize("dtype,case,opts", [
    ("f64", _steady(1), {}), ("f32", _steady(3), {}), ("f64", _unsteady(2), {}), ("f32", _unsteady(1), {}),
    ("f64", _steady(2), {"mf": 1}), ("f32", _steady(2), {"mf": 2}), ("f64", _unsteady(1), {"mf": 2, "dp": 2}),
    ("f64", _steady(1), {"recon": 4, "opsplit": 2}), ("f32", _unsteady(2), {"recon": 2, "opsplit": 3, "mt": 2}),
    ("f64", _unsteady(1), {"recon": 1, "dp": 2, "opsplit": 2})])
def test_steps_that_fill_their_own_ghosts(N, tile, dtype, case, opts):
    one = _run(N, case, [1] * 13, dtype=dtype, tile=tile, **opts)
    _same(_run(N, case, [2, 7, 1, 3], dtype=dtype, tile=tile, **opts), one)
    _same(_run(N, case, [9, 4], graph=4, dtype=dtype, tile=tile, **opts), one)


@pytest.mark.parametrize("N", [13, 61, 130])
@pytest.mark.parametrize("opts", [{}, {"dp": 2}, {"opsplit": 2}, {"opsplit": 3, "mt": 2}, {"recon": 1},
                                  {"recon": 2, "dp": 2}, {"recon": 4, "opsplit": 2, "dp": 2}])
def test_flux_tables_have_the_bits_of_formed_weights(N, opts, monkeypatch):
    from cubedsphere.solver import Advection
    with_table = _run(N, _steady(2), [5], **opts)
    monkeypatch.setattr(Advection, "bind_flux_tables", staticmethod(lambda *a, **k: None))
    _same(_run(N, _steady(2), [5], **opts), with_table)


@pytest.mark.parametrize("change", ["dt", "recon", "opsplit"])
def test_flux_tables_of_another_step_are_left_out(change, monkeypatch):
    from cubedsphere.solver import Advection

    def run():
        sol = Advection(21, _steady(1), 0.01, device="cuda:0", max_steps=8).init_vars_adv()
        sol.step(3)
        if change == "dt":
            sol.dt *= 0.5
        else:
            sol.opts["recon" if change == "recon" else "split"] = 2
        sol.refresh()
        sol.step(3)
        out = sol.full_state()
        sol.close()
        return out

    with_table = run()
    monkeypatch.setattr(Advection, "bind_flux_tables", staticmethod(lambda *a, **k: None))
    assert np.array_equal(with_table, run())


@pytest.mark.parametrize("dp,dtype", [(1, "f64"), (2, "f64"), (2, "f32")])
def test_steady_and_unsteady_solves_in_one_handle(dp, dtype):
    from cubedsphere.batch import Batch, make_members
    specs = [(19, _steady(1), 6), (24, _unsteady(3), 6), (33, _steady(2), 6), (12, _unsteady(1), 6)]
    batch = Batch(make_members(specs, dtype=dtype, dp=dp), graph_steps=3).init()
    batch.step(6)
    for k, spec in enumerate(specs):
        alone = Batch(make_members([spec], dtype=dtype, dp=dp), graph_steps=0).init()
        alone.step(6)
        assert np.array_equal(batch.members[k].full_state(), alone.members[0].full_state()), k
        alone.close()
    batch.close()


# 400: the four tracers are two launches
@pytest.mark.parametrize("N,dtype,et,mf", [(13, "f64", 1, 1), (24, "f64", 2, 2), (48, "f64", 2, 3), (13, "f32", 2, 3),
                                           (33, "f32", 1, 2), (400, "f64", 1, 3)])
def test_general_step_tracers_together_and_alone(N, dtype, et, mf):
    from cubedsphere.cases import Case
    case = _unsteady(4)
    together = _run(N, case, [2, 1], dtype=dtype, et=et, mf=mf)
    for t in range(case.ntr):
        alone = _run(N, Case([case.tracers[t]], case.wind), [2, 1], dtype=dtype, et=et, mf=mf)
        assert np.array_equal(together[1][t], alone[1][0]) and together[2][t] == alone[2][0], t


@pytest.mark.parametrize("n", [0, 1, 131071, 131072, 524287, 524288, 524289, 1500001])
def test_read_out_through_staging(n):
    from cubedsphere.solver import to_host
    t = torch.arange(2 * n, device="cuda:0", dtype=torch.float64)[::2]
    assert np.array_equal(to_host(t), t.cpu().numpy())
