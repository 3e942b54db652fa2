"""Searches with Johnson LB2 over the forms of its walk: one to three chunks of
64 machine pairs, both sides of 32 jobs, one machine pair, a pool whose layout
is larger than its instances.  The incumbent is frozen (no schedule is below
it), so every count is a whole number that equals the CPU oracle's.
"""
import pytest

pytestmark = pytest.mark.gpu

# jobs, machines, incumbent
TREES = [(3, 2, 231), (12, 16, 1529), (32, 5, 1780), (32, 12, 2324), (32, 13, 2328), (33, 12, 2302), (33, 13, 2326),
         (32, 17, 2493), (32, 20, 2896), (33, 20, 2749)]


def _counts(r):
    return r.decomposed, r.leaves, r.simple_bounds, r.johnson_bounds


def _config(mode):
    return dict(bound_mode=mode[0], branching=mode[1], refine=1, johnson_pairs=0)


@pytest.mark.parametrize("mode", [(2, 3), (1, 1)])
@pytest.mark.parametrize("n,m,ub", TREES)
def test_search_counts(oracle_mod, n, m, ub, mode):
    import pbbperm_amd as P
    O = oracle_mod
    ptm = O.synth_ptm(77, n, m)
    want = _counts(O.solve(ptm, ub, **_config(mode)))
    for team in (0, 8192):
        cfg = P.default_config(nb_ivms=1024, early_stop_johnson=0, team_nodes=team, **_config(mode))
        with P.GpuBB(ptm, cfg, ub=ub) as eng:
            assert eng.solve(time_budget=60.0)
            assert _counts(eng.stats()) == want


@pytest.mark.parametrize("jobs,machines", [(32, 20), (33, 13), (33, 20)])
def test_pool_counts(oracle_mod, jobs, machines):
    import pbbperm_amd as P
    import pbbperm_amd.pool as PP
    O = oracle_mod
    trees = [t for t in TREES if t[0] <= jobs and t[1] <= machines]
    ptms = [O.synth_ptm(77, n, m) for n, m, _ in trees]
    ubs = [ub for _, _, ub in trees]
    want = [_counts(O.solve(p, ub, **_config((2, 3)))) for p, ub in zip(ptms, ubs)]
    with PP.Pool(P.default_config(early_stop_johnson=0, **_config((2, 3))), max_jobs=jobs, machines=machines, slots=16,
                 waves_per_group=4, explorers_per_instance=64) as pool:
        res, _ = pool.solve(ptms, ubs, time_budget=60.0)
    assert [_counts(r) for r in res] == want
