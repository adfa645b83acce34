"""The FP64 fitting in one call (csrc/fit_chain.hip): row counts around the 16-,
32- and 64-row tiles, empty types, every resnet form, narrow and wide layers,
against torch's FP64 autograd on the CPU."""

import numpy as np
import pytest
import torch

from deepmd_amd import model as M

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _torch_energy(layers, d):
    x = d
    for ly in layers[:-1]:
        y = torch.tanh(x @ torch.tensor(ly.w) + torch.tensor(ly.b))
        if ly.idt is not None:
            y = y * torch.tensor(ly.idt)
        r = M._res_mode(ly.w.shape[0], ly.w.shape[1], ly.resnet)
        x = y + (x if r == 1 else torch.cat([x, x], -1) if r == 2 else 0.0)
    return (x @ torch.tensor(layers[-1].w))[:, 0] + float(layers[-1].b[0])


@pytest.mark.parametrize("widths,d3,m2,rows,dt,chain", [
    ([240, 240, 240], 100, 16, [27, 54], True, True),      # 16 x 16 tiles, K split
    ([240, 240, 240], 100, 16, [513, 1000], True, True),   # 32 x 32 tiles
    ([240, 240], 128, 16, [5000], False, True),            # 64 x 64 tiles
    ([32, 64, 64], 64, 4, [1, 0, 17], True, True),         # resnet 2 and 1, an empty type
    ([16], 32, 8, [33], False, True),                      # one layer
    ([48, 48, 96], 40, 16, [16, 15, 2], True, True),
    ([256, 256, 256], 128, 16, [64, 65], False, True),
    ([240, 240], 32, 4, [5493], True, True),               # the line of width 256
    ([240, 240], 32, 4, [5494], True, False),              # beyond: the library's products
    ([512, 512], 32, 4, [1300, 1500], False, False),
    ([64, 64], 24, 4, [12000], True, True),
])
def test_fit_chain_vs_autograd(widths, d3, m2, rows, dt, chain):
    rng = np.random.default_rng(5)
    nt = len(rows)
    nets = [M._layers(M._rand_net(rng, [d3 * m2] + widths + [1], dt, True)) for _ in range(nt)]
    bias = rng.normal(size=nt)
    fit = M.Fitting(nets, bias, np.zeros(nt), "f64", torch.device(DEV))
    assert fit.chain is not None
    n = sum(rows)
    order = rng.permutation(n).astype(np.int32)
    segs = [(t, sum(rows[:t]), sum(rows[:t + 1])) for t in range(nt)]
    xyz = rng.normal(size=(n, 4, d3)) * 0.3
    x = torch.tensor(xyz, device=DEV)
    ae = torch.full((n,), float("nan"), dtype=torch.float64, device=DEV)
    gx = torch.full((n, 4, d3), float("nan"), dtype=torch.float64, device=DEV)
    bf = fit.buffers(n)
    assert ("ws" in bf) == chain
    fit.run(ae, gx, x, torch.tensor(order, device=DEV), segs, n, bf, d3, m2,
            torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    ref = torch.tensor(xyz, requires_grad=True)
    e = torch.zeros(n, dtype=torch.float64)
    for t, a, b in segs:
        if b == a:
            continue
        idx = torch.tensor(order[a:b].astype(np.int64))
        xs = ref[idx]
        d = torch.matmul(xs.transpose(1, 2), xs[:, :, :m2]).reshape(b - a, -1)
        e = e.index_put((idx,), _torch_energy(nets[t], d) + bias[t])
    g, = torch.autograd.grad(e.sum(), ref)
    # sums of up to 2048 terms rounded at 1.1e-16, through a few layers: < 1e-12
    # of the largest value
    for name, got, want in (("energy", ae, e.detach()), ("gxyz", gx, g)):
        err = float((got.cpu() - want).abs().max() / want.abs().max())
        print(f"{name} {widths} {rows}: {err:.2e}", flush=True)
        assert err < 1e-12, name


@pytest.mark.parametrize("rows", [[20, 30], [700, 1400]])  # K split over the wavefronts, 32 x 32
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_fit_chain_not_finite(rows, bad):
    """A slot that is not finite stays alone: the others' energies and gradients
    are what they are without it, bit for bit."""
    rng = np.random.default_rng(6)
    nets = [M._layers(M._rand_net(rng, [100 * 16, 240, 240, 1], True, True)) for _ in rows]
    fit = M.Fitting(nets, np.zeros(2), np.zeros(2), "f64", torch.device(DEV))
    n = sum(rows)
    segs = [(0, 0, rows[0]), (1, rows[0], n)]
    order = torch.arange(n, dtype=torch.int32, device=DEV)
    xyz = rng.normal(size=(n, 4, 100)) * 0.3
    at = rows[0] - 1  # the last row of a type, which tiles beyond the end read again
    out = []
    for v in (xyz[at, 1, 3], bad):
        xyz[at, 1, 3] = v
        ae = torch.zeros(n, dtype=torch.float64, device=DEV)
        gx = torch.zeros((n, 4, 100), dtype=torch.float64, device=DEV)
        bf = fit.buffers(n)
        assert "ws" in bf
        fit.run(ae, gx, torch.tensor(xyz, device=DEV), order, segs, n, bf, 100, 16,
                torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        out.append((ae.cpu().numpy(), gx.cpu().numpy()))
    keep = np.arange(n) != at
    for a, b in zip(*out):
        assert np.array_equal(a[keep], b[keep])
    assert not np.isfinite(out[1][1][at]).all()


def test_fit_chain_rows_of_present_types():
    """The form is chosen by the rows of the types that have slots, not by the
    number of nets; both forms give the same energies there."""
    rng = np.random.default_rng(7)
    h, d3, m2, nx = 512, 8, 4, M.Fitting.chain_rows(512)
    n = int(nx) + 40
    nets = [M._layers(M._rand_net(rng, [d3 * m2, h, h, 1], True, True)) for _ in range(2)]
    fit = M.Fitting(nets, np.zeros(2), np.zeros(2), "f64", torch.device(DEV))
    one, two = [(0, 0, n), (1, n, n)], [(0, 0, n // 2), (1, n // 2, n)]
    assert "ws" not in fit.buffers(n, one)
    assert "ws" in fit.buffers(n, two) and "ws" in fit.buffers(n)
    assert "ws" in fit.buffers(n - 40, one) and "ws" in fit.buffers(1, [(0, 0, 0), (1, 0, 0)])
    order = torch.arange(n, dtype=torch.int32, device=DEV)
    xyz = torch.tensor(rng.normal(size=(n, 4, d3)) * 0.3, device=DEV)
    out = []
    for bf in (fit.buffers(n, one), fit.buffers(n)):
        ae = torch.zeros(n, dtype=torch.float64, device=DEV)
        gx = torch.zeros((n, 4, d3), dtype=torch.float64, device=DEV)
        fit.run(ae, gx, xyz, order, one, n, bf, d3, m2, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        out.append((ae.cpu().numpy(), gx.cpu().numpy()))
    for a, b in zip(*out):
        # sums of at most 512 FP64 products a layer, four layers' depth
        assert np.abs(a - b).max() <= 512 * 4 * 2.3e-16 * max(np.abs(b).max(), 1.0)
