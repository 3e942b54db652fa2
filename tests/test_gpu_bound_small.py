"""The batched bounds of small batches, a schedule per wavefront: the edges of a
tile of four schedules, both sides of the largest such batch, the smallest and
largest shapes, malformed schedules among the others, against the CPU oracle (whole
numbers, equal)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(3, 2), (33, 17), (63, 20)])
@pytest.mark.parametrize("count", [2, 3, 4, 5, 255, 4096, 4097])
def test_small_batches_match_oracle(oracle_mod, n, m, count):
    import torch
    import pbbperm_amd as P
    O = oracle_mod
    ptm = O.synth_ptm(47, n, m)
    perms, l1, l2 = O.random_partials(n, max(count, 64), 5, edge_frac=0.3)
    perms, l1, l2 = perms[:count].copy(), l1[:count].copy(), l2[:count].copy()
    ref = O.Instance(ptm).bounds_batch(perms, l1, l2, which=("cb", "ce", "lb1n", "lb2", "mk"))
    bad, off = np.zeros(count, bool), np.zeros(count, bool)
    perms[1, 1] = perms[1, 0]  # a repeated job
    bad[1] = True
    if count > 3:
        l1[count - 1], l2[2] = -2, n + 1
        off[[2, count - 1]] = True
    dev = [torch.from_numpy(np.ascontiguousarray(x, dtype=np.int32)).cuda() for x in (perms, l1, l2)]
    b = P.Bounds(ptm)
    cb, ce = b.lb1_children(*dev)
    got = dict(cb=cb, ce=ce, lb1n=b.lb1_node(*dev), lb2=b.lb2_node(*dev), mk=b.makespan(dev[0]))
    for name, value in got.items():
        want = ref[name].copy()
        want[bad if name == "mk" else bad | off] = -1
        np.testing.assert_array_equal(value.cpu().numpy(), want, err_msg=name)
