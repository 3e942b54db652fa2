"""Johnson LB2 searches of instances with times above the packed table's limit (a
small instance's times 12-fold, which keeps its tree): the wide table in LDS, where
fewer explorers are resident than the engine has, and in global memory, where the
intervals do not fit those.  The incumbent is frozen, so every count is a whole
number that equals the CPU oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SCALE = 12
# jobs, machines, incumbent of the unscaled instance: one to three chunks of 64
# pairs, both sides of 32 jobs, the largest table
TREES = [(3, 2, 231), (12, 16, 1529), (32, 5, 1780), (32, 12, 2324), (33, 12, 2287), (32, 20, 2894), (33, 20, 2743),
         (63, 20, 4253)]


def _counts(r):
    return r.decomposed, r.leaves, r.simple_bounds, r.johnson_bounds


def _config(mode):
    return dict(bound_mode=mode[0], branching=mode[1], refine=1, johnson_pairs=0)


def _instance(O, n, m):
    ptm = np.ascontiguousarray(O.synth_ptm(77, n, m) * SCALE)
    assert ptm.max() > 1023
    return ptm


@pytest.mark.parametrize("mode", [(2, 3), (1, 1)])
@pytest.mark.parametrize("n,m,ub", TREES)
def test_search_counts(oracle_mod, n, m, ub, mode):
    import pbbperm_amd as P
    ptm = _instance(oracle_mod, n, m)
    want = _counts(oracle_mod.solve(ptm, ub * SCALE, **_config(mode)))
    for team in (0, 8192):
        cfg = P.default_config(nb_ivms=1 << 14, early_stop_johnson=0, team_nodes=team, **_config(mode))
        with P.GpuBB(ptm, cfg, ub=ub * SCALE) as eng:
            assert eng.solve(time_budget=60.0)
            assert _counts(eng.stats()) == want


@pytest.mark.parametrize("n,m,ub", [t for t in TREES if t[0] > 30 and t[1] == 20])
def test_intervals_of_the_last_explorers(oracle_mod, n, m, ub):
    """An interval each for the engine's last explorers, past those that are
    resident with the table in LDS: every explorer is launched, and the search
    goes on from there as from the first ones.  The path down to an interval's
    first node is bounded but not counted, so the oracle's count is that of the
    same intervals."""
    import pbbperm_amd as P
    mode = (2, 3)
    ptm = _instance(oracle_mod, n, m)
    cfg = P.default_config(nb_ivms=1 << 14, early_stop_johnson=0, team_nodes=100, team_waves=4, **_config(mode))
    with P.GpuBB(ptm, cfg, ub=ub * SCALE) as eng:
        eng.init_full_interval()
        assert not eng.next(node_budget=100)
        ids, pos, end, _, _ = eng.get_intervals()
        E = eng.stats().explorers
        assert 0 < len(ids) < E
        want = sum(oracle_mod.solve(ptm, ub * SCALE, pos=p, end=e, **_config(mode)).decomposed for p, e in zip(pos, end))
        for first in (E - len(ids), 0):
            eng.init_from_fac(np.arange(first, first + len(ids)), pos, end)
            assert eng.next(time_budget=60.0)
            assert eng.stats().decomposed == want


def test_replay_of_one_shape_in_both_forms(oracle_mod):
    """One engine per shape: packed and wide instances take turns in it."""
    import pbbperm_amd as P
    import pbbperm_amd.pool as PP
    ptms, best = [], []
    for i in range(6):
        ptm = oracle_mod.synth_ptm(300 + i, 11, 12)
        opt = oracle_mod.solve(ptm, oracle_mod.Instance(ptm).neh()[0]).best
        k = SCALE if i % 2 else 1
        ptms.append(np.ascontiguousarray(ptm * k))
        best.append(opt * k)
    assert [p.max() > 1023 for p in ptms] == [False, True] * 3
    cfg = P.default_config(nb_ivms=1 << 14, early_stop_johnson=0, **_config((2, 3)))
    res, _, _ = PP.plain_replay(ptms, [PP.UB_NEH] * 6, np.zeros(6), cfg, time_budget=60.0)
    assert [r.status for r in res] == ["solved"] * 6
    assert [r.best for r in res] == best


@pytest.mark.parametrize("jobs,machines", [(12, 16), (32, 20), (33, 12)])
def test_pool_counts(oracle_mod, jobs, machines):
    """Both forms in one pool: tables that fit the layout's LDS and that do not."""
    import pbbperm_amd as P
    import pbbperm_amd.pool as PP
    trees = [t for t in TREES if t[0] <= jobs and t[1] <= machines]
    ptms = [_instance(oracle_mod, n, m) for n, m, _ in trees] + [oracle_mod.synth_ptm(77, n, m) for n, m, _ in trees]
    ubs = [ub * SCALE for _, _, ub in trees] + [ub for _, _, ub in trees]
    want = [_counts(oracle_mod.solve(p, ub, **_config((2, 3)))) for p, ub in zip(ptms, ubs)]
    with PP.Pool(P.default_config(early_stop_johnson=0, **_config((2, 3))), max_jobs=jobs, machines=machines, slots=16,
                 waves_per_group=4, explorers_per_instance=64) as pool:
        res, _ = pool.solve(ptms, ubs, time_budget=60.0)
    assert [_counts(r) for r in res] == want
