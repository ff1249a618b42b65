"""Batches beyond the last-level cache, stepped in groups of grids: every grid
ends on the bits and shifter of stepping it alone, whatever the group borders
(grids larger than a group, several in one group, the run's parity of steps)."""
import numpy as np
import pytest

from periodicshiftlbm_amd import cases

pytestmark = pytest.mark.gpu

# 16-bit: 270 MB (a group of its own), 27 MB, 95 MB, 101 MB and 1 MB
EDGES = (136, 63, 96, 98, 21)


# two grids beyond the cache next to each other (278 and 284 MB, one group) and one apart
EDGES_BEYOND = (136, 30, 137, 138, 60)


# box-face cells from the lists (FP16), in the bulk launch (BF16, FP32), fused; calls that step
# in groups, and calls of too few steps for it (BF16 3, fused FP16 3)
@pytest.mark.parametrize("storage,tuning,order,steps", [("f16", 4, 0, 2), ("bf16", 4, 1, 5), ("f16", 12, 0, 3),
                                                        ("f16", 12, 0, 6), ("f32", 4, 1, 4), ("bf16", 4, 0, 3)])
def test_grouped_batch_equals_single_grid_steps(psl, storage, tuning, order, steps):
    _check(psl, EDGES, storage, tuning, order, steps)


@pytest.mark.parametrize("storage,tuning,order,steps", [("bf16", 4, 0, 4), ("bf16", 4, 1, 4), ("f16", 12, 1, 6),
                                                        ("f16", 4, 0, 3)])
def test_grids_beyond_the_cache_in_one_group(psl, storage, tuning, order, steps):
    _check(psl, EDGES_BEYOND, storage, tuning, order, steps)


def _check(P, edges, storage, tuning, order, steps):
    doms = [{"shape": (2 * L, L, L), "nu": 1e-3 * (1 + i), "u_inlet": 0.04, "diameter": 0.25 * L,
             "center": (0.5 * L,) * 3} for i, L in enumerate(edges)]
    batched = [cases.domain_grid(d, storage)[0] for d in doms]
    assert sum(54 * g.n for g in batched) > 2 * 192 << 20
    b = P.Batch(batched)
    b.set_tuning(tuning, order)
    b.step(steps)
    b.step(1)
    b.step(steps + 1)
    for d, g in zip(doms, batched):
        alone = cases.domain_grid(d, storage)[0]
        P.updateGrid([alone], 2 * steps + 2)
        assert g.shifter.tolist() == alone.shifter.tolist()
        nbad = int(np.count_nonzero(g.get_f().view(np.uint32) != alone.get_f().view(np.uint32)))
        assert nbad == 0, f"{d['shape']}: {nbad} values differ"
        alone.close()
    b.close()
    for g in batched:
        g.close()
