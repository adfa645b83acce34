"""Row-wise force and virial additions of the operators (csrc/force_virial.hip,
add_rows): row lengths around a wavefront, empty entries and entries outside
the region, against the oracle."""

import numpy as np
import pytest
import torch

from oracle import cops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("nf,nloc,nall,nnei", [(1, 1, 1, 1), (2, 5, 9, 63), (1, 7, 7, 64),
                                               (2, 6, 40, 65), (1, 9, 20, 130)])
def test_force_virial_rows(nf, nloc, nall, nnei):
    import deepmd_amd.ops  # noqa: F401
    rng = np.random.default_rng(nnei)
    nl = rng.integers(-1, nall, (nf, nloc, nnei)).astype(np.int32)
    nd = rng.normal(size=(nf, nloc * nnei * 4))
    ed = rng.normal(size=(nf, nloc, nnei * 12))
    rij = rng.normal(size=(nf, nloc, nnei * 3))
    to = lambda a: torch.tensor(a, device=DEV)  # noqa: E731
    f = torch.ops.deepmd.prod_force_se_a(to(nd), to(ed), to(nl), nloc, nall)
    v, av = torch.ops.deepmd.prod_virial_se_a(to(nd), to(ed), to(rij), to(nl), nloc, nall)
    # entries outside the region add nothing to any row
    out = np.where(rng.random(nl.shape) < 0.1, nall + 3, nl).astype(np.int32)
    v2, av2 = torch.ops.deepmd.prod_virial_se_a(to(nd), to(ed), to(rij), to(out), nloc, nall)
    f2 = torch.ops.deepmd.prod_force_se_a(to(nd), to(ed), to(out), nloc, nall)
    rv, rav = cops.prod_virial_a(nd, ed, rij, nl, nall)
    rv2, rav2 = cops.prod_virial_a(nd, ed, rij, np.where(out >= nall, -1, out), nall)
    rf = cops.prod_force_a(nd, ed, nl, nall)
    # (the centre's own row takes every slot's share, listed neighbour or not)
    rf2 = cops.prod_force_a(nd, ed, np.where(out >= nall, -1, out), nall)
    # sums of at most nloc nnei products rounded at 1.1e-16
    for got, ref in ((f, rf), (f2, rf2), (v, rv), (av, rav), (v2, rv2), (av2, rav2)):
        ref = ref.reshape(got.shape)
        assert np.max(np.abs(got.cpu().numpy() - ref)) <= 1e-13 * max(np.max(np.abs(ref)), 1.0)
