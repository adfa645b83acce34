"""Neighbour search and forces where several workgroups share a cell's centres
(few cells, or frames of different sizes): the lists against the per-centre
search's, entry by entry, and forces and virial against the per-slot kernel's."""

import numpy as np
import pytest
import torch

from deepmd_amd.model import SeAModel, random_model_dict

pytestmark = pytest.mark.gpu
DEV = "cuda"
NLIST_MODE, FORCE_MODE = 0, 2  # DPK_TUNE_* keys of include/dpk.h


def _frame(n, edge, seed):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    x = (g[rng.permutation(len(g))[:n]] + 0.5) * edge / m + rng.uniform(-0.2, 0.2, (n, 3))
    return x, rng.integers(0, 2, n).astype(np.int32), np.diag([edge] * 3)


@pytest.mark.parametrize("sizes", [
    [(1, 5.0)], [(16, 7.0)], [(17, 7.0)], [(81, 9.3)], [(130, 9.9)],       # one cell
    [(400, 16.0)], [(1000, 21.0)],                                       # 27 and 64 cells
    [(24, 7.2), (43, 7.0), (90, 11.0), (300, 17.0), (7, 6.0)],           # one batch
    [(81, 9.3)] * 4, [(192, 12.4)] * 33,                                 # frames of one size
    [(400, 16.0)] * 12, [(60, 9.0), (100, 9.5), (80, 9.2)],              # (the last divides too)
])
def test_shared_cells(sizes):
    d = random_model_dict(3, 5.0, 0.5, [60, 60], [25, 50, 100], 16, [32, 32])
    frames = [_frame(n, e, 5 + k) for k, (n, e) in enumerate(sizes)]
    out = []
    for mode in (0, 1):  # cell workgroups; a wavefront a centre and a slot's own atomics
        m = SeAModel(d, "f64", DEV)
        m.tuning.set(NLIST_MODE, mode)
        m.tuning.set(FORCE_MODE, mode)
        s = m.system([f[0] for f in frames], [f[1] for f in frames],
                     [f[2].reshape(9) for f in frames], nlocs=[len(f[1]) for f in frames])
        r = m.evaluate(s, atomic_virial=True)
        torch.cuda.synchronize()
        out.append((s.nlist.cpu().numpy().copy(),
                    {k: v.cpu().numpy().copy() for k, v in r.items()}))
    assert np.array_equal(out[0][0], out[1][0])
    for k, ref in out[1][1].items():
        # FP64 sums of up to 120 slots in another order
        assert np.max(np.abs(out[0][1][k] - ref)) <= 1e-12 * max(np.max(np.abs(ref)), 1e-30), k
