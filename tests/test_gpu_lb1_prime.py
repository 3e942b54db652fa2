"""Searches with the LB1' refinement in every branching mode (back and alternate
branching prune on it alone: their back-direction LB1 costs stay zero), on both
sides of 32 children: counts under a frozen incumbent are whole numbers and
equal the CPU oracle's.
"""
import pytest

pytestmark = pytest.mark.gpu


# trees that the oracle does not finish within its node limit are left out
@pytest.mark.parametrize("bound_mode", [1, 2])
@pytest.mark.parametrize("branching", [-3, -2, -1, 1, 2, 3])
def test_counts_of_every_branching(oracle_mod, bound_mode, branching):
    import pbbperm_amd as P
    O = oracle_mod
    done = 0
    for seed, n, m in [(3, 8, 5), (5, 9, 20), (2, 30, 10), (3, 61, 19), (3, 33, 2)]:
        ptm = O.synth_ptm(seed, n, m)
        neh, _ = O.Instance(ptm).neh()
        ub = O.solve(ptm, neh).best if n < 10 else {30: 2105, 61: 4029, 33: int(ptm.sum(1).max())}[n]
        mode = dict(bound_mode=bound_mode, branching=branching, refine=0)
        ref = O.solve(ptm, ub, max_nodes=60000, **mode)
        if ref.decomposed >= 60000:
            continue
        done += 1
        with P.GpuBB(ptm, P.default_config(nb_ivms=512, **mode), ub=ub) as eng:
            assert eng.solve(time_budget=60.0)
            st = eng.stats()
        assert (st.decomposed, st.leaves, st.simple_bounds, st.johnson_bounds) == (
            ref.decomposed, ref.leaves, ref.simple_bounds, ref.johnson_bounds), (seed, n, m)
    assert done >= 2
