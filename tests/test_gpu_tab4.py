"""Tabulated embedding with four basis functions (csrc/tabulate.hip, k_tab4_fwd /
k_tab4_bwd): channel counts below, at and above what one and two channels a
lane hold, odd ones, tables that are not aligned, rows with and without
padding, values outside the table, blocks of one slot and over 64; operator and
fused form, against the oracle's restatement."""

import numpy as np
import pytest
import torch

from oracle import cops

pytestmark = pytest.mark.gpu
DEV = "cuda"
# 300 slots x 6 terms (and 200 channels x 4) rounded at eps, of the largest
# value: < 1e3 eps
TOL = {torch.float64: 1e3 * 2.3e-16, torch.float32: 1e3 * 1.2e-7}


def _inputs(nloc, nnei, L, dt, seed, pad=True):
    rng = np.random.default_rng(seed)
    nrow = 120
    table = rng.normal(size=(nrow, 6 * L)) * np.tile([1, 1, .5, .2, .1, .05], L)
    info = np.array([-1.0, 5.0, 11.0, 0.1, 0.1, -1.0])  # 60 + 60 intervals
    x = np.sort(rng.uniform(-1.3, 12.0, size=(nloc, nnei)), axis=1)[:, ::-1].copy()
    em = rng.normal(size=(nloc, nnei, 4))
    em[..., 0] = x
    if pad:
        for i in range(nloc):
            n = (0, nnei, nnei - 1)[i] if i < 3 else rng.integers(0, nnei + 1)
            em[i, n:] = [-0.5, 0, 0, 0]
    npdt = np.float64 if dt == torch.float64 else np.float32
    dy = rng.normal(size=(nloc, 4, L))
    return [a.astype(npdt) for a in (table, info, em, dy)]


def _rel(a, b):
    return np.max(np.abs(a.astype(np.float64) - b)) / np.max(np.abs(b))


@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
@pytest.mark.parametrize("nloc,nnei,L,shift,pad", [
    (5, 92, 100, 0, True), (1, 1, 1, 0, False), (6, 65, 63, 0, True), (6, 64, 64, 0, False),
    (4, 130, 128, 0, True), (3, 20, 130, 0, True), (3, 20, 101, 0, True), (3, 20, 200, 1, True),
    (3, 20, 100, 2, True), (4, 300, 60, 0, True),
])
def test_tab4_operator(nloc, nnei, L, shift, pad, dt):
    import deepmd_amd.ops  # noqa: F401
    table, info, em, dy = _inputs(nloc, nnei, L, dt, 3 + L, pad)
    buf = torch.empty(table.size + 4, dtype=dt, device=DEV)
    tt = buf[shift:shift + table.size].view(table.shape)  # shift: unaligned rows
    tt.copy_(torch.from_numpy(table))
    e = torch.tensor(em, device=DEV, requires_grad=True)
    ex = e.detach()[..., 0].reshape(-1, 1).contiguous().requires_grad_(True)
    out = torch.ops.deepmd.tabulate_fusion_se_a(tt, torch.from_numpy(info), ex, e, L)[0]
    dx, dem = torch.autograd.grad(out, (ex, e), torch.tensor(dy, device=DEV))
    t64, i64, em64, dy64 = (a.astype(np.float64) for a in (table, info, em, dy))
    # the interval of a value is found in the table's precision
    ref = cops.tabulate_fusion_se_a(table, info, em[..., :1].reshape(-1, 1), em, L)
    rdx, rdem = cops.tabulate_fusion_se_a_grad(table, info, em[..., :1].reshape(-1, 1), em, dy)
    tol = TOL[dt]
    for name, a, b in (("out", out, ref), ("dx", dx, rdx), ("dem", dem, rdem)):
        err = _rel(a.detach().cpu().numpy().reshape(b.shape), b.astype(np.float64))
        print(f"{name} {nloc}x{nnei}x{L} shift {shift} {dt}: {err:.2e}", flush=True)
        assert err < tol, name


@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
@pytest.mark.parametrize("sel,L", [([46, 92], 100), ([5, 70, 1], 60), ([130], 33)])
def test_tab4_fused(sel, L, dt):
    """The fused form: a table a type block, folds per block, xyz / nnei."""
    from deepmd_amd._lib import DPK_PREC_F32, DPK_PREC_F64, call, ptr, stream_ptr
    from deepmd_amd.model import ctypes_array, ctypes_int_array
    nt, nnei, n = len(sel), sum(sel), 9
    parts = [_inputs(n, s, L, dt, 11 + k) for k, s in enumerate(sel)]
    em = np.concatenate([p[2] for p in parts], axis=1)
    gx = parts[0][3]
    tables = torch.tensor(np.concatenate([p[0].ravel() for p in parts]), device=DEV)
    offs = np.cumsum([0] + [p[0].size for p in parts])[:-1]
    off, nsp = ctypes_array(offs, "longlong"), ctypes_int_array([p[0].shape[0] for p in parts])
    inf = ctypes_array(np.concatenate([p[1] for p in parts]).astype(np.float64), "double")
    sec = ctypes_int_array(np.concatenate([[0], np.cumsum(sel)]))
    at = torch.zeros(n, dtype=torch.int32, device=DEV)
    net_of = torch.arange(nt, dtype=torch.int32, device=DEV).repeat(nt)
    e, g = torch.tensor(em, device=DEV), torch.tensor(gx, device=DEV)
    xyz = torch.empty((n, 4, L), dtype=dt, device=DEV)
    nd = torch.full((n, nnei, 4), float("nan"), dtype=dt, device=DEV)
    prec = DPK_PREC_F64 if dt == torch.float64 else DPK_PREC_F32
    tail = (ptr(tables), off[1], nsp[1], inf[1], ptr(net_of), nt, nt, sec[1], L, n, nnei,
            stream_ptr())
    call("dpk_tab_embed_fwd", ptr(xyz), prec, ptr(e), ptr(at), *tail)
    call("dpk_tab_embed_bwd", ptr(nd), prec, ptr(e), ptr(g), ptr(at), *tail)
    torch.cuda.synchronize()
    ref, rnd = 0.0, []
    for p in parts:
        x = p[2][..., :1].reshape(-1, 1)
        ref = ref + cops.tabulate_fusion_se_a(p[0], p[1], x, p[2], L).astype(np.float64) / nnei
        dx, dem = cops.tabulate_fusion_se_a_grad(p[0], p[1], x, p[2], gx)
        dem = dem.astype(np.float64)
        dem[..., 0] += dx.reshape(dem.shape[:2])
        rnd.append(dem / nnei)
    assert _rel(xyz.cpu().numpy(), ref) < TOL[dt]
    assert _rel(nd.cpu().numpy(), np.concatenate(rnd, axis=1)) < TOL[dt]
