"""The times the iteration callback reports, with and without a replayed
graph, for a caller that times only those (profile_kinds "iter")."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("variant", [1, 3])
def test_every_iteration_has_its_sweep_time(variant, graph):
    """A replayed iteration is reported whole as sweep time: positive in every
    iteration, and all of them within the loop's time."""
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = D.gen_uniform(700, 400, 20000, 500, seed=3)
    k = 4
    with S.Solver(0) as s:
        s.upload(ds)
        for _ in range(2):  # a second run replays the graph of the first
            recs = []
            s.set_factors(D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32))
            s.run(k, 0.05, 4, 2, variant=variant, use_graph=graph, profile=True, profile_kinds=("iter",),
                  callback=recs.append)
            assert len(recs) == 4
            assert all(r.rank_time > 0 and r.rmse_time > 0 for r in recs)
            assert graph or all(r.update_time > 0 for r in recs)
            assert s.loop_time() >= sum(r.rank_time + r.update_time + r.rmse_time for r in recs)


def test_one_call_reports_times_under_a_graph():
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = D.gen_uniform(700, 400, 20000, 500, seed=3)
    param = S.Parameter()
    param.use_graph, param.maxiter = 1, 3
    lines = []
    S.cdmf_ocl_02(ds, D.initial_col(param.k, ds.m), np.zeros((param.k, ds.n), np.float32), ds, param, log=lines.append)
    assert len(lines) == 3
    sums = [float(x.split("rank_time")[1].split("|")[1].split()[0]) for x in lines]
    # 0.1 ms steps: ten ranks of ten sweeps each take longer
    assert 0 < sums[0] < sums[1] < sums[2], lines
