"""The batched bounds at the edges of their tiles (16 to 128 schedules), on the
smallest and largest shapes, with malformed schedules among the others, against
the CPU oracle (whole numbers, equal)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(3, 2), (20, 10), (63, 20)])
@pytest.mark.parametrize("count", [1, 15, 17, 8193, 70001])
def test_tiles_match_oracle(oracle_mod, n, m, count):
    import torch
    import pbbperm_amd as P
    O = oracle_mod
    ptm = O.synth_ptm(31, n, m)
    perms, l1, l2 = O.random_partials(n, max(count, 64), 9, edge_frac=0.1)
    perms, l1, l2 = perms[:count], l1[:count], l2[:count]
    ref = O.Instance(ptm).bounds_batch(perms, l1, l2, which=("cb", "ce", "cbf", "lb1n", "lb2", "mk"))
    perms, l1, l2 = perms.copy(), l1.copy(), l2.copy()
    bad = np.zeros(count, bool)  # a bad order
    off = np.zeros(count, bool)  # a bad front or back
    if count > 1:
        perms[0, n - 1], perms[3, 0], perms[5, 1] = n, -1, perms[5, 0]
        bad[[0, 3, 5]] = True
        l1[7], l2[9], l2[11], l1[count - 1] = -2, n + 1, l1[11], n
        off[[7, 9, 11, count - 1]] = True
    dev = [torch.from_numpy(np.ascontiguousarray(x, dtype=np.int32)).cuda() for x in (perms, l1, l2)]
    b = P.Bounds(ptm)
    cb, ce = b.lb1_children(*dev)
    cbf, _ = b.lb1_children(*dev, both=False)
    got = dict(cb=cb, ce=ce, cbf=cbf, lb1n=b.lb1_node(*dev), lb2=b.lb2_node(*dev), mk=b.makespan(dev[0]))
    for name, value in got.items():
        want = ref[name].copy()
        want[bad if name == "mk" else bad | off] = -1
        np.testing.assert_array_equal(value.cpu().numpy(), want, err_msg=name)
