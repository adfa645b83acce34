"""Tabulated embedding with four basis functions (csrc/tabulate.hip, k_tab4_fwd /
k_tab4_bwd / k_tab4_bwd_narrow): channel counts below, at and above what one and
two channels a lane hold, odd and narrow ones, tables that are not aligned, rows
with and without padding, values outside the table, blocks of one slot and over
64, one, two, four and eight wavefronts an atom in the backward; operator and
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
    (5, 92, 8, 0, True), (3, 20, 16, 0, False), (4, 64, 32, 0, True), (4, 63, 32, 0, True),
    (4, 70, 17, 1, True), (7, 200, 33, 0, True), (3, 150, 300, 0, True), (3, 70, 257, 0, True),
    (1000, 40, 48, 0, True), (1030, 33, 66, 0, True), (2040, 34, 40, 0, True),
    (2050, 34, 40, 0, True), (500, 130, 36, 0, True),
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
@pytest.mark.parametrize("sel,L,n", [([46, 92], 100, 9), ([5, 70, 1], 60, 9), ([130], 33, 9),
                                     ([46, 92], 16, 40), ([5, 70, 1], 32, 700)])
def test_tab4_fused(sel, L, n, dt):
    """The fused form: a table for every centre type and type block (atoms of
    all types, virtual ones as type 0), folds per block, xyz / nnei."""
    from deepmd_amd._lib import DPK_PREC_F32, DPK_PREC_F64, call, ptr, stream_ptr
    from deepmd_amd.model import ctypes_array, ctypes_int_array
    nt, nnei = len(sel), sum(sel)
    at = np.random.default_rng(L).integers(-1, nt, n).astype(np.int32)
    ti = np.maximum(at, 0)
    # table (block k, centre type c) is net k nt + c; rows and dE/dxyz are shared
    parts = [[_inputs(n, s, L, dt, 11 + k + 7 * c) for c in range(nt)] for k, s in enumerate(sel)]
    em = np.concatenate([p[0][2] for p in parts], axis=1)
    gx = parts[0][0][3]
    flat = [q for p in parts for q in p]
    tables = torch.tensor(np.concatenate([q[0].ravel() for q in flat]), device=DEV)
    offs = np.cumsum([0] + [q[0].size for q in flat])[:-1]
    off, nsp = ctypes_array(offs, "longlong"), ctypes_int_array([q[0].shape[0] for q in flat])
    inf = ctypes_array(np.concatenate([q[1] for q in flat]).astype(np.float64), "double")
    sec = ctypes_int_array(np.concatenate([[0], np.cumsum(sel)]))
    net_of = torch.tensor([k * nt + c for c in range(nt) for k in range(nt)], dtype=torch.int32,
                          device=DEV)
    e, g, a = (torch.tensor(v, device=DEV) for v in (em, gx, at))
    xyz = torch.empty((n, 4, L), dtype=dt, device=DEV)
    nd = torch.full((n, nnei, 4), float("nan"), dtype=dt, device=DEV)
    prec = DPK_PREC_F64 if dt == torch.float64 else DPK_PREC_F32
    tail = (ptr(tables), off[1], nsp[1], inf[1], ptr(net_of), nt, nt * nt, sec[1], L, n, nnei,
            stream_ptr())
    call("dpk_tab_embed_fwd", ptr(xyz), prec, ptr(e), ptr(a), *tail)
    call("dpk_tab_embed_bwd", ptr(nd), prec, ptr(e), ptr(g), ptr(a), *tail)
    torch.cuda.synchronize()
    ref, rnd = np.zeros((n, 4, L)), []
    for p in parts:
        rows = p[0][2]
        dblk = np.zeros(rows.shape)
        for c in range(nt):
            m = ti == c
            if not m.any():
                continue
            x = rows[m][..., :1].reshape(-1, 1)
            ref[m] += cops.tabulate_fusion_se_a(p[c][0], p[c][1], x, rows[m], L).astype(
                np.float64) / nnei
            dx, dem = cops.tabulate_fusion_se_a_grad(p[c][0], p[c][1], x, rows[m], gx[m])
            dem = dem.astype(np.float64)
            dem[..., 0] += dx.reshape(dem.shape[:2])
            dblk[m] = dem / nnei
        rnd.append(dblk)
    assert _rel(xyz.cpu().numpy(), ref) < TOL[dt]
    assert _rel(nd.cpu().numpy(), np.concatenate(rnd, axis=1)) < TOL[dt]


@pytest.mark.parametrize("L", [16, 100])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_tab4_not_finite(L, bad):
    """A value that is not finite stays in its atom (and reads inside the
    table): the others' results are what they are without it, bit for bit."""
    import deepmd_amd.ops  # noqa: F401
    table, info, em, dy = _inputs(12, 70, L, torch.float32, 5)
    out = []
    for v in (em[4, 0, 0], bad):
        em[4, 0, 0] = v
        e = torch.tensor(em, device=DEV, requires_grad=True)
        ex = e.detach()[..., 0].reshape(-1, 1).contiguous().requires_grad_(True)
        o = torch.ops.deepmd.tabulate_fusion_se_a(torch.tensor(table, device=DEV),
                                                  torch.from_numpy(info), ex, e, L)[0]
        dx, dem = torch.autograd.grad(o, (ex, e), torch.tensor(dy, device=DEV))
        out.append([t.detach().cpu().numpy().reshape(12, -1) for t in (o, dx, dem)])
    keep = np.arange(12) != 4
    for a, b in zip(*out):
        assert np.array_equal(a[keep], b[keep])
    assert not np.isfinite(out[1][0][4]).all()
