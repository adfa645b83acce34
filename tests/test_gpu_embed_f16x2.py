"""FP16X2 embedding kernels (csrc/embed_f16x2.hip) on their own, against the
oracle's descriptor contraction and its autograd: resnet and time-step variants,
nets in LDS and read from memory, block lengths around the 16-slot tile, four,
two and one wavefronts an atom (the limits are 512 and 1,536 atoms on 256 CUs)."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from deepmd_amd.model import SeAModel, random_model_dict
from oracle import sea

pytestmark = pytest.mark.gpu
DEV = "cuda"

# The weights are FP16 values (below), so what is left is the split operands'
# 2^-22 and FP32's tanh (1e-7), grown by a factor of about two a layer, and FP32
# sums of up to 200 slots, whose errors average out: below 2e-6 of the largest
# value; a lost low part would be 2^-11 = 5e-4.
TOL = 2e-6
K = 2.8853900817779268  # the kernels' weights are rounded after this scaling


def _case(neuron, sel, one_side, natoms, dt, seed=5):
    d = random_model_dict(seed, 6.0, 0.5, sel, neuron, 4, [16, 16], type_one_side=one_side,
                          resnet_dt_emb=dt, activation="tanh", fitting_activation="tanh")
    de = d["model"]["descriptor"]
    nt, nnei = len(sel), sum(sel)
    rng = np.random.default_rng(seed + 1)
    davg = np.zeros((nt, nnei, 4))
    davg[..., 0] = 0.3 * (1 + np.arange(nt)[:, None])
    de["@variables"]["davg"]["value"] = davg.tolist()
    de["@variables"]["dstd"]["value"] = np.full((nt, nnei, 4), 0.5).tolist()
    for net in de["embeddings"]["networks"]:
        for ly in net["layers"][1:]:
            w = ly["@variables"]["w"]
            h = (np.asarray(w["value"], np.float32) * np.float32(K)).astype(np.float16)
            w["value"] = (h.astype(np.float64) / K).tolist()
    at = rng.integers(0, nt, natoms).astype(np.int32)
    em = rng.normal(size=(natoms, nnei, 4)).astype(np.float32)
    nl = np.zeros((natoms, nnei), dtype=np.int32)
    sec = np.concatenate([[0], np.cumsum(sel)])
    for i in range(natoms):
        for t in range(nt):
            real = rng.integers(0, sel[t] + 1) if i > 2 else (sel[t], 0, sel[t] // 2)[i]
            nl[i, sec[t] + real:sec[t + 1]] = -1
            em[i, sec[t] + real:sec[t + 1]] = -davg[at[i], 0] / 0.5
    gx = (1e-3 * rng.normal(size=(natoms, 4, neuron[-1]))).astype(np.float32)
    return d, at, em, nl, gx


@pytest.mark.parametrize("neuron,sel,one_side,natoms,dt", [
    ([25, 50, 100], [46, 92], True, 7, False),      # two nets in LDS
    ([32, 64, 128], [200], True, 1100, False),
    ([25, 50, 100], [17, 15], False, 41, False),    # four nets, read from memory
    ([25, 50, 100], [16], True, 1, True),
    ([10, 20, 40], [1, 31], True, 9, True),
    ([20, 30, 100], [40], True, 50, False),         # no doubling: no resnet
    ([20, 40, 100], [33], True, 4300, False),       # resnet of layer 2 only
    ([25, 50, 100], [20, 33], True, 512, False),    # the last with four wavefronts an atom
    ([25, 50, 100], [20, 33], False, 513, False),   # the first with two
    ([25, 50, 100], [3, 30], True, 1536, True),     # the last with two
    ([25, 50, 100], [3, 30], True, 1537, True),
    ([25, 50, 100], [17], True, 100, False),        # two tiles: two wavefronts at most
    ([20, 50, 100], [15, 16, 17], False, 30, True),  # of layer 3 only, nine nets
])
def test_embed_f16x2_vs_oracle(neuron, sel, one_side, natoms, dt):
    d, at, em, nl, gx = _case(neuron, sel, one_side, natoms, dt)
    om = sea.model_from_serialized(d)
    e = torch.tensor(em, dtype=torch.float64, requires_grad=True)
    _, xyz = sea.descriptor_from_env(om, e, torch.tensor(at).long(),
                                     torch.ones(em.shape[:2], dtype=torch.int32))
    nd, = torch.autograd.grad((xyz * torch.tensor(gx)).sum(), e)
    nd = np.where((nl < 0)[..., None], 0.0, nd.numpy())
    m = SeAModel(d, "f16x2", DEV)
    to = lambda a: torch.tensor(a, device=DEV).contiguous()  # noqa: E731
    nan = lambda *s: torch.full(s, float("nan"), device=DEV)  # noqa: E731
    s = SimpleNamespace(fs=SimpleNamespace(natoms=natoms), em=to(em), atype=to(at), nlist=to(nl),
                        gxyz=to(gx), xyz=nan(natoms, 4, m.d3), nd=nan(*em.shape))
    st = torch.cuda.current_stream().cuda_stream
    m._embed_forward(s, st)
    m._embed_backward(s, st)
    torch.cuda.synchronize()
    for got, ref, what in ((s.xyz, xyz.detach().numpy(), "xyz"), (s.nd, nd, "net_deriv")):
        err = np.max(np.abs(got.cpu().numpy() - ref)) / np.max(np.abs(ref))
        print(f"{what} {neuron} {sel} n={natoms}: {err:.2e}", flush=True)
        assert err < TOL, what


# Rounding at the scale of the operands: with weights that are FP16 values and
# tangents split at one to two times the derivatives themselves, a value or a
# tangent keeps 2^-22 of itself and at worst 2^-25 absolute (FP16's subnormals);
# the second decides where weights are small and no resnet copy holds the
# derivatives up.  2-norms of the error over the result's: (xyz, net_deriv, ds),
# a third above what kernels that split tanh and the tangents at this scale
# reach on these cases.
SMALL = {
    ((32, 64, 128), 1.0): (2.2e-7, 3.1e-7, 3.8e-7),
    ((32, 64, 128), 0.3): (2.2e-7, 3.1e-7, 5.0e-7),
    ((32, 64, 128), 0.1): (2.4e-7, 3.1e-7, 1.3e-6),
    ((20, 30, 100), 1.0): (2.2e-7, 3.3e-7, 4.2e-7),
    ((20, 30, 100), 0.3): (3.6e-7, 4.0e-7, 1.6e-6),
    ((20, 30, 100), 0.1): (4.0e-7, 4.1e-7, 3.2e-5),
    ((20, 40, 100), 0.1): (3.6e-7, 4.0e-7, 2.8e-6),
    ((20, 50, 100), 0.1): (3.6e-7, 4.8e-7, 9.6e-6),
}


@pytest.mark.parametrize("neuron,scale", list(SMALL))
@pytest.mark.parametrize("natoms", [64, 1600])
def test_embed_f16x2_operand_bits(neuron, scale, natoms):
    """Errors of the split operands alone, also for small weights, and of the
    radial derivative ds apart from dE/dR (gx without its first component)."""
    d, at, em, nl, gx = _case(list(neuron), [60], True, natoms, False)
    rng = np.random.default_rng(9)
    de = d["model"]["descriptor"]
    de["@variables"]["davg"]["value"] = np.zeros((1, 60, 4)).tolist()
    for net in de["embeddings"]["networks"]:
        for k, ly in enumerate(net["layers"]):
            w = ly["@variables"]["w"]
            v = np.asarray(w["value"]) * scale
            v = (v * K).astype(np.float16).astype(np.float64) / K if k else v.astype(np.float32)
            w["value"] = np.asarray(v, np.float64).tolist()
    em = rng.normal(size=em.shape).astype(np.float32)
    nl = np.zeros_like(nl)
    om = sea.model_from_serialized(d)
    m = SeAModel(d, "f16x2", DEV)
    to = lambda a: torch.tensor(a, device=DEV).contiguous()  # noqa: E731
    err = []
    for first in (1.0, 0.0):
        gx = gx.copy()
        gx[:, 0] *= first
        e = torch.tensor(em, dtype=torch.float64, requires_grad=True)
        _, xyz = sea.descriptor_from_env(om, e, torch.tensor(at).long(),
                                         torch.ones(em.shape[:2], dtype=torch.int32))
        nd, = torch.autograd.grad((xyz * torch.tensor(gx)).sum(), e)
        s = SimpleNamespace(fs=SimpleNamespace(natoms=natoms), em=to(em), atype=to(at),
                            nlist=to(nl), gxyz=to(gx), nd=torch.zeros(*em.shape, device=DEV),
                            xyz=torch.zeros(natoms, 4, m.d3, device=DEV))
        st = torch.cuda.current_stream().cuda_stream
        m._embed_forward(s, st)
        m._embed_backward(s, st)
        torch.cuda.synchronize()
        pairs = ((s.xyz, xyz.detach()), (s.nd, nd)) if first else ((s.nd[..., 0], nd[..., 0]),)
        err += [float((g.cpu().double() - r).norm() / r.norm()) for g, r in pairs]
    print(f"{neuron} x {scale} n={natoms}: " + " ".join(f"{v:.2e}" for v in err), flush=True)
    assert all(v < t for v, t in zip(err, SMALL[neuron, scale])), err


@pytest.mark.parametrize("natoms", [40, 700, 1700])  # four, two and one wavefronts an atom
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_embed_f16x2_not_finite(natoms, bad):
    """A row that is not finite stays in its atom: the others' results are what
    they are without it, bit for bit."""
    d, at, em, nl, gx = _case([25, 50, 100], [20, 33], True, natoms, False)
    nl[4, 0] = 0
    m = SeAModel(d, "f16x2", DEV)
    to = lambda a: torch.tensor(a, device=DEV).contiguous()  # noqa: E731
    out = []
    for v in (em[4, 0, 0], bad):
        em[4, 0, 0] = v
        s = SimpleNamespace(fs=SimpleNamespace(natoms=natoms), em=to(em), atype=to(at),
                            nlist=to(nl), gxyz=to(gx), nd=torch.zeros(*em.shape, device=DEV),
                            xyz=torch.zeros(natoms, 4, m.d3, device=DEV))
        st = torch.cuda.current_stream().cuda_stream
        m._embed_forward(s, st)
        m._embed_backward(s, st)
        torch.cuda.synchronize()
        out.append((s.xyz.cpu().numpy(), s.nd.cpu().numpy()))
    keep = np.arange(natoms) != 4
    for a, b in zip(*out):
        assert np.array_equal(a[keep], b[keep])
    assert not np.isfinite(out[1][0][4]).all() and not np.isfinite(out[1][1][4, 0]).all()
