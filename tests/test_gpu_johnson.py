"""The Johnson tables' two forms (packed words up to a time of 1023, pairs of
words above) in LDS and in global memory, against the CPU oracle: bounds are
whole numbers and equal it exactly.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dev(*arrs):
    import torch
    return [torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda() for a in arrs]


# both sides of the 32-job mask, the largest n; one pair, tables on both sides of the LDS limit; both sides of the packed
# form's largest time, the largest time an instance may hold
@pytest.mark.parametrize("top", [99, 1023, 1024, 1000000])
@pytest.mark.parametrize("n,m", [(3, 2), (32, 20), (33, 14), (33, 20), (63, 13), (63, 20)])
def test_lb2_over_table_forms(oracle_mod, n, m, top):
    import pbbperm_amd as P
    O = oracle_mod
    ptm = O.synth_ptm(77, n, m).astype(np.int64) * top // 99
    ptm[0, 0], ptm[m - 1, n - 1], ptm[m // 2, 0] = top, top, 0
    ptm = ptm.astype(np.int32)
    perms, l1, l2 = O.random_partials(n, 700, 5, edge_frac=0.1)
    b = P.Bounds(ptm)
    dev = _dev(perms, l1, l2)
    for pairs in (0, 1, 2):
        ref = O.Instance(ptm).bounds_batch(perms, l1, l2, pairs=pairs, which=("lb2",))["lb2"]
        np.testing.assert_array_equal(b.lb2_node(*dev, pairs).cpu().numpy(), ref)


@pytest.mark.parametrize("mode", [(2, 3), (1, 1)])
def test_searches_on_large_times(oracle_mod, mode):
    """All times and the incumbent times 20 (above the packed form's limit):
    every bound scales, so the search is the same."""
    import pbbperm_amd as P
    import pbbperm_amd.pool as PP
    O = oracle_mod
    bm, br = mode
    cfg = dict(bound_mode=bm, branching=br, refine=1, johnson_pairs=0, early_stop_johnson=0)
    ptms = [O.synth_ptm(900 + i, 10 + i % 3, 5) for i in range(8)]
    opts = [O.solve(p, O.Instance(p).neh()[0]).best for p in ptms]
    refs = [O.solve(p, o, bound_mode=bm, branching=br, refine=1) for p, o in zip(ptms, opts)]
    want = [(r.decomposed, r.leaves, r.simple_bounds, r.johnson_bounds) for r in refs]
    for p, o, w in zip(ptms, opts, want):
        with P.GpuBB(p * np.int32(20), P.default_config(nb_ivms=256, **cfg), ub=20 * o) as eng:
            assert eng.solve(time_budget=60.0)
            st = eng.stats()
        assert (st.decomposed, st.leaves, st.simple_bounds, st.johnson_bounds) == w
    # small and large times side by side in one pool
    both = [p * np.int32(20) if i % 2 else p for i, p in enumerate(ptms)]
    ubs = [20 * o if i % 2 else o for i, o in enumerate(opts)]
    with PP.Pool(P.default_config(**cfg), max_jobs=12, machines=5, slots=8, waves_per_group=2,
                 explorers_per_instance=64) as pool:
        res, _ = pool.solve(both, ubs, time_budget=60.0)
    assert [(r.decomposed, r.leaves, r.simple_bounds, r.johnson_bounds) for r in res] == want
