"""FP64 embedding kernels (csrc/embed_f64.hip) on their own, against the oracle's
descriptor contraction and its autograd: nets in LDS together and in groups,
seven and eight channel steps, one wavefront an atom and several (few atoms),
block lengths around the 16-slot tile, and the padding left out or not."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from deepmd_amd.model import SeAModel, random_model_dict
from oracle import sea

pytestmark = pytest.mark.gpu
DEV = "cuda"

# error of a sum of 200 slots of products through three layers of at most 64
# terms, each rounded at 1.1e-16 (and the tanh to a few of these): < 1e-13 of
# the largest value; with a margin of ten
TOL = 1e-12


def _case(neuron, sel, one_side, natoms, act="tanh", dt=False, scale=1.0, avg=0.3, seed=3):
    d = random_model_dict(seed, 6.0, 0.5, sel, neuron, 4, [16, 16], type_one_side=one_side,
                          resnet_dt_emb=dt, activation=act, fitting_activation="tanh")
    de = d["model"]["descriptor"]
    nt, nnei = len(sel), sum(sel)
    rng = np.random.default_rng(seed + 1)
    davg = np.zeros((nt, nnei, 4))
    davg[..., 0] = avg * (1 + np.arange(nt)[:, None])
    de["@variables"]["davg"]["value"] = davg.tolist()
    de["@variables"]["dstd"]["value"] = np.full((nt, nnei, 4), 0.5).tolist()
    for net in de["embeddings"]["networks"]:
        for ly in net["layers"]:
            w = ly["@variables"]["w"]
            w["value"] = (np.asarray(w["value"]) * scale).tolist()
    at = rng.integers(0, nt, natoms).astype(np.int32)
    em = rng.normal(size=(natoms, nnei, 4))
    nl = np.zeros((natoms, nnei), dtype=np.int32)
    sec = np.concatenate([[0], np.cumsum(sel)])
    for i in range(natoms):
        for t in range(nt):
            real = rng.integers(0, sel[t] + 1) if i > 2 else (0, sel[t], sel[t] // 2)[i]
            nl[i, sec[t] + real:sec[t + 1]] = -1
            em[i, sec[t] + real:sec[t + 1]] = -davg[at[i], 0] / 0.5
    gx = rng.normal(size=(natoms, 4, neuron[-1]))
    return d, at, em, nl, gx


def _run(d, at, em, nl, gx, skip):
    m = SeAModel(d, "f64", DEV)
    m.skip_padding = skip
    n = len(at)
    to = lambda a: torch.tensor(a, device=DEV).contiguous()  # noqa: E731
    s = SimpleNamespace(fs=SimpleNamespace(natoms=n), em=to(em), atype=to(at), nlist=to(nl),
                        gxyz=to(gx), xyz=torch.full((n, 4, m.d3), float("nan"), device=DEV,
                                                    dtype=torch.float64),
                        nd=torch.full(em.shape, float("nan"), device=DEV, dtype=torch.float64))
    st = torch.cuda.current_stream().cuda_stream
    m._embed_forward(s, st)
    m._embed_backward(s, st)
    torch.cuda.synchronize()
    return s.xyz.cpu().numpy(), s.nd.cpu().numpy()


def _oracle(d, at, em, gx):
    om = sea.model_from_serialized(d)
    e = torch.tensor(em, requires_grad=True)
    mask = torch.ones(em.shape[:2], dtype=torch.int32)
    _, xyz = sea.descriptor_from_env(om, e, torch.tensor(at).long(), mask)
    nd, = torch.autograd.grad((xyz * torch.tensor(gx)).sum(), e)
    return xyz.detach().numpy(), nd.numpy()


def _check(got, ref, what):
    err = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
    print(f"{what}: {err:.2e}", flush=True)
    assert err < TOL, what


@pytest.mark.parametrize("neuron,sel,one_side,natoms,extra", [
    ([25, 50, 100], [46, 92], True, 7, {}),           # two nets in LDS, eight wavefronts an atom
    ([25, 50, 100], [46, 92], True, 1100, {}),        # two nets in LDS, one wavefront an atom
    ([25, 50, 100], [17, 15], False, 40, {}),         # four nets, two at a time
    ([28, 56, 112], [16], True, 1, {}),               # the widest of seven steps
    ([29, 58, 116], [33], True, 130, {}),             # the narrowest of eight
    ([32, 64, 128], [200], True, 600, {}),
    ([10, 20, 40], [1, 31], True, 9, {}),
    ([32, 64, 128], [20, 20], True, 30, {}),          # two wide nets, one at a time
    ([25, 50, 100], [30], True, 50, {"act": "gelu"}),
    ([25, 50, 100], [30, 20], True, 50, {"act": "silut:2.5", "dt": True}),
    ([20, 30, 100], [40], True, 50, {}),              # no doubling: no resnet copies
    ([25, 50, 100], [46], True, 50, {"scale": 40.0}),  # saturated activations
])
def test_embed_f64_vs_oracle(neuron, sel, one_side, natoms, extra):
    d, at, em, nl, gx = _case(neuron, sel, one_side, natoms, **extra)
    xyz, nd = _oracle(d, at, em, gx)
    for skip in (True, False):
        x, n = _run(d, at, em, nl, gx, skip)
        _check(x, xyz, f"xyz {neuron} {sel} n={natoms} skip={skip}")
        _check(n, nd, f"net_deriv {neuron} {sel} n={natoms} skip={skip}")


def test_embed_f64_padding_rows_that_differ():
    """Statistics that vary over the slots: padding rows with their own
    derivative each."""
    d, at, em, nl, gx = _case([25, 50, 100], [40, 20], True, 30, avg=0.0)
    davg = np.random.default_rng(0).normal(size=(2, 60, 4)) * 0.2
    d["model"]["descriptor"]["@variables"]["davg"]["value"] = davg.tolist()
    em = np.where((nl < 0)[..., None], -davg[at] / 0.5, em)
    xyz, nd = _oracle(d, at, em, gx)
    x, n = _run(d, at, em, nl, gx, True)
    _check(x, xyz, "xyz")
    _check(n, nd, "net_deriv")


def test_embed_f64_nan_and_infinity():
    """A NaN stays in its atom; an infinite slot saturates the net as torch's
    tanh does, and what its infinite row makes of the sums is not finite in the
    same places (the resnet copy is summed apart, so inf - inf can be a NaN
    where the oracle has an infinity)."""
    d, at, em, nl, gx = _case([32, 64, 128], [30], True, 20)
    em[4, 0, 0] = np.nan
    nl[4] = 0
    x, n = _run(d, at, em, nl, gx, True)
    assert np.isnan(x[4]).all() and np.isnan(n[4, 0, 0])
    keep = np.arange(20) != 4
    assert np.isfinite(x[keep]).all() and np.isfinite(n[keep]).all()
    em[4, 0] = [np.inf, 1.0, 1.0, 1.0]
    x, _ = _run(d, at, em, nl, gx, True)
    ref, _ = _oracle(d, at, em, gx)
    assert np.array_equal(np.isfinite(x[4]), np.isfinite(ref[4]))
    _check(x[4, 1:], ref[4, 1:], "components with a finite row")


@pytest.mark.parametrize("neuron,sel,one_side,natoms,extra", [
    ([32, 64, 128], [20, 9, 14], False, 61, {}),      # nine nets: a workgroup lists those it uses
    ([25, 50, 100], [17, 15], False, 2100, {}),       # more atoms than wavefronts
    ([32, 64, 128], [33, 18], True, 1100, {}),        # all atoms in both groups, whole and split
    ([32, 64, 128], [33, 18], True, 300, {}),
    ([32, 64, 128], [2, 3], False, 16500, {}),        # more than 64 atoms a workgroup
    ([10, 20, 40], [2] * 16, False, 90, {}),          # 256 nets, the most there can be
    ([20, 30, 100], [30, 20], False, 700, {"dt": True}),
    ([25, 50, 100], [30, 20], False, 600, {"act": "gelu"}),
])
def test_embed_f64_nets_in_groups(neuron, sel, one_side, natoms, extra):
    """Nets that don't fit in LDS together; every seventh atom is virtual (its
    rows are zero and its list is empty: zero in the forward, the derivative of
    type 0 in the backward)."""
    d, at, em, nl, gx = _case(neuron, sel, one_side, natoms, **extra)
    em[3::7], nl[3::7] = 0.0, -1
    real = at.copy()
    at[3::7], real[3::7] = -1, 0
    xyz, nd = _oracle(d, real, em, gx)
    for skip in (True, False):
        x, n = _run(d, at, em, nl, gx, skip)
        _check(x, xyz, f"xyz {neuron} {sel} n={natoms} skip={skip}")
        _check(n, nd, f"net_deriv {neuron} {sel} n={natoms} skip={skip}")
        assert not x[3::7].any()
