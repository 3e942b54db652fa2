"""A Johnson table in LDS costs no explorers: an engine takes as many intervals
with LB2 as three workgroups per CU hold, at the shapes where the table would fill
the CU's LDS as at the smallest and largest ones."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(3, 2), (58, 14), (59, 14), (63, 14), (54, 15), (58, 15), (49, 16), (51, 16), (43, 17),
                                 (45, 17), (40, 18), (32, 20), (63, 20)])
def test_lb2_explorers_at_the_lds_limit(n, m):
    import numpy as np
    import torch

    import pbbperm_amd as P
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    most = 3 * 4 * cus
    cfg = P.default_config(nb_ivms=1 << 16, bound_mode=2, branching=3, refine=1, johnson_pairs=0, early_stop_johnson=0)
    assert P.explorers_for(n, m, cfg) >= most
    # whatever the times: 12-fold they are past the packed table's limit
    with P.GpuBB(P.synth(n + m, n, m) * 12, cfg, ub=0) as eng:
        assert eng.stats().explorers == P.explorers_for(n, m, cfg)
    # so many intervals are taken, the last explorers among their ids
    with P.GpuBB(P.synth(n + m, n, m), cfg, ub=0) as eng:
        E = eng.stats().explorers
        ids = np.arange(E - most, E)
        pos = np.zeros((most, n), np.intc)
        eng.init_from_fac(ids, pos, pos)
        assert eng.stats().active == most
