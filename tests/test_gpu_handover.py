"""Hand-overs between explorers: the idle mask (words of 64 explorers) and the
self-tagged messages of the mailboxes.

With the incumbent frozen, the decomposed nodes do not depend on how intervals
are handed on, so every explorer count and every sequence of stopped launches
must give the oracle's counts.  A launch that stops on its node budget leaves
messages at explorers that had gone already; they have to come back as
intervals of the saved state, exported and resumed like any other.
"""
import pytest

pytestmark = pytest.mark.gpu


def _want(ref):
    return (ref.best, ref.decomposed, ref.leaves, ref.simple_bounds, ref.johnson_bounds)


def _got(eng):
    st = eng.stats()
    return (eng.best()[0], st.decomposed, st.leaves, st.simple_bounds, st.johnson_bounds)


# edges of the mask words (one explorer, one word less one, full, plus one; two words and a bit of a third), 63 jobs (the
# largest ids and positions of a message), 20 machines (the largest stack entries) and few of both
@pytest.mark.parametrize("nb", [1, 63, 64, 65, 129])
@pytest.mark.parametrize("seed,n,m,ub,mode", [
    (3, 63, 20, 4230, dict(bound_mode=0, branching=1)),
    (2, 30, 10, 2117, dict(bound_mode=0, branching=1)),
    (3, 18, 5, None, dict(bound_mode=2, branching=3, refine=1, johnson_pairs=0, early_stop_johnson=0)),
])
def test_counts_over_word_edges_and_stopped_launches(oracle_mod, seed, n, m, ub, mode, nb):
    import pbbperm_amd as P
    O = oracle_mod
    ptm = O.synth_ptm(seed, n, m)
    if ub is None:
        ub = O.solve(ptm, O.Instance(ptm).neh()[0]).best
    ref = O.solve(ptm, ub, bound_mode=mode["bound_mode"], branching=mode["branching"], refine=mode.get("refine", 0))
    cfg = P.default_config(nb_ivms=nb, team_nodes=0, steal_margin=1, **mode)
    with P.GpuBB(ptm, cfg, ub=ub) as eng:
        assert eng.solve(time_budget=60.0)
        assert _got(eng) == _want(ref)
        # the same search again in short launches
        eng.init_full_interval()
        runs = 1
        while not eng.next(node_budget=200, time_budget=60.0):
            runs += 1
            assert runs < 10000
        assert _got(eng) == _want(ref)


def _number(digits):
    value, n = 0, len(digits)
    for i, d in enumerate(digits):
        value = value * (n - i) + int(d)
    return value


def test_intervals_of_a_stopped_launch_are_disjoint(oracle_mod):
    """What a stopped launch saves, messages under way among it, is one interval
    per active explorer, none empty and no two overlapping."""
    import pbbperm_amd as P
    O = oracle_mod
    ptm = O.synth_ptm(2, 30, 10)
    cfg = P.default_config(nb_ivms=256, team_nodes=0, steal_margin=1, bound_mode=0, branching=1)
    with P.GpuBB(ptm, cfg, ub=2117) as eng:
        eng.init_full_interval()
        for _ in range(8):
            done = eng.next(node_budget=300, time_budget=60.0)
            ids, pos, end, _, _ = eng.get_intervals()
            assert len(ids) == eng.stats().active
            if done:
                break
            spans = sorted((_number(b), _number(e)) for b, e in zip(pos, end))
            assert all(b <= e for b, e in spans)
            assert all(e < b for (_, e), (b, _) in zip(spans, spans[1:]))
