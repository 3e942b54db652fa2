"""team_nodes holds a search in the team (explorers 0-15 with LB1, 0-7 with a
refinement bound) for as many nodes as the caller set, and a run for fewer nodes
stops in the team near its budget: it has saved intervals of those explorers only.
Incumbent frozen, so the whole search's count is exact."""
import pytest

pytestmark = pytest.mark.gpu

LB2 = dict(bound_mode=2, branching=1, refine=1, johnson_pairs=0, early_stop_johnson=0)
LB1 = dict(bound_mode=0, branching=1)

# mode, team size, seed, jobs, machines, incumbent, nodes of the tree, node budget of the first run
SEARCHES = [(LB2, 8, 1, 20, 10, 1548, 3636, 2500), (LB1, 16, 2, 30, 10, 2117, 5394, 4700)]


@pytest.mark.parametrize("mode,team,seed,n,m,ub,nodes,budget", SEARCHES)
@pytest.mark.parametrize("team_nodes", [5000, 100000, 8192])
def test_team_keeps_a_search_for_team_nodes(mode, team, seed, n, m, ub, nodes, budget, team_nodes):
    import pbbperm_amd as P
    cfg = P.default_config(nb_ivms=4096, team_nodes=team_nodes, **mode)
    with P.GpuBB(P.synth(seed, n, m), cfg, ub=ub) as eng:
        eng.init_full_interval()
        assert not eng.next(node_budget=budget)
        ids = eng.get_intervals()[0]
        assert len(ids) and max(ids) < team
        # an explorer looks at the budget every 64 nodes
        assert budget <= eng.stats().decomposed < budget + 64 * team
        assert eng.next()
        assert eng.stats().decomposed == nodes


def test_a_search_that_improves_its_incumbent_stays_with_the_team(oracle_mod):
    """From NEH, at the default: a few explorers find the optimum of this tree and
    prove it within a quarter of team_nodes, which the team then has; thousands of
    them search twice as many before the same schedules prune them."""
    import pbbperm_amd as P
    cfg = P.default_config(nb_ivms=4096, bound_mode=2, branching=3, refine=1, johnson_pairs=0, early_stop_johnson=0)
    ptm = P.synth(0, 20, 5)
    ub, order = P.neh(ptm)
    with P.GpuBB(ptm, cfg, ub=ub, ub_perm=order) as eng:
        assert eng.solve(time_budget=60.0)
        best, _ = eng.best()
        assert best < ub and eng.stats().decomposed < cfg.team_nodes // 4 + 64 * 8
        assert best == oracle_mod.solve(ptm, best + 1).best
