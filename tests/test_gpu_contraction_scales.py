"""GPU tests of the contraction (contraction.hpp) where an operand's largest values do not count:
tokens or outputs without a gradient, inputs and outputs whose two thresholds are equal, gradients of
different magnitudes, rows far below threshold; and tables of other shapes than the transistor's.
Every output is compared with float64 against its own scale, the root of the sum of its cells' squares.

Bounds. Formula: the operands carry 2^-24 of each value (16 terms' pairs and singles and the truncated
series 2.5e-7, measured in float64 arithmetic), sums add up to sqrt(n / 2) 2^-25 for n slabs of 16
elements (2e-7 at the 250 here); four times their sum, 2e-6, for the largest of a few thousand groups.
Table: a row's lookups in fp32 are off by 5e-6 to 1.5e-5 of their differences (coordinates of up to 4096
records round to 2^-13 of a record); what the harmonics leave out is below that, and the largest group is
held to 2e-5.
"""

from __future__ import annotations

import pytest
import torch

from tests.helpers import flash_cfg, oracle_tables
from tests.test_gpu_contraction import PARAMS, V_SAT

pytestmark = pytest.mark.gpu

TOL = {"formula": 2e-6, "table": 2e-5}
SHAPE = {"formula": (3700, 192, 768), "table": (2048, 384, 1536)}  # 2^29 and 2^30 cells
SPREAD = 0.2142


def _formula_cells(v):
    n, u_t, i_s, v_d = PARAMS
    a = 1.0 / (2.0 * n * u_t)

    def sp(u):
        return torch.nn.functional.softplus(u, threshold=40.0)

    u1, u2 = v * a, (v - v_d) * a
    s1, s2 = sp(u1), sp(u2)
    return i_s * (s1 * s1 - s2 * s2), i_s * 2.0 * a * (s1 * torch.sigmoid(u1) - s2 * torch.sigmoid(u2))


def _table_cells(ti, td, lo, hi):
    n = ti.numel()
    ti, td = ti.double().cuda(), td.double().cuda()

    def cells(v):
        c = ((v - lo) * ((n - 1) / (hi - lo))).clamp(0, n - 1)
        i = c.floor().clamp(max=n - 2).long()
        f = c - i
        return tuple(t[i] + f * (t[i + 1] - t[i]) for t in (ti, td))

    return cells


def _reference(x, wp, wn, g, cells):
    """(out, dX, dVth+, dVth-) in float64 and their scales."""
    xd, pd, nd, gd = (t.double() for t in (x, wp, wn, g))
    vals = [torch.zeros_like(t) for t in (gd, xd, pd, nd)]
    sums = [torch.zeros_like(t) for t in (gd, xd, pd, nd)]
    step = max(1, int(1e7 // wp.numel()))
    for a in range(0, x.shape[0], step):
        b = slice(a, a + step)
        r, gb = 1.0 / (1.0 + xd[b, None, :] / V_SAT), gd[b, :, None]
        ip, sp = cells(xd[b, None, :] - pd[None])
        inn, sn = cells(xd[b, None, :] - nd[None])
        for q, (cell, dims) in enumerate((((ip - inn) * r, 2), (gb * ((sp - sn) * r - (ip - inn) * r * r / V_SAT), 1),
                                          (-gb * sp * r, 0), (gb * sn * r, 0))):
            if q < 2:
                vals[q][b] = cell.sum(dims)
                sums[q][b] = cell.square().sum(dims)
            else:
                vals[q] += cell.sum(dims)
                sums[q] += cell.square().sum(dims)
    return vals, [s.sqrt() for s in sums]


def _tables(cfg):
    from isa.approximations.delta_lut import lut_range
    from isa.kernels.transformer_ffn import _hip, ops

    lo, hi, n = lut_range(cfg)
    ti, td = (torch.as_tensor(t) for t in oracle_tables(cfg))
    packed = [ops.pack_tables(ti.cuda(), td.cuda(), layout) for layout in (_hip.LUT_FWD, _hip.LUT_BWD)]
    return packed, n, lo, hi, _table_cells(ti, td, lo, hi)


def _run(kind, x, wp, wn, g, tables=None, took=(True, True)):
    """took: whether the contraction has to take the forward and the backward (None: either)."""
    from isa.kernels.transformer_ffn import ops

    (M, K), O = x.shape, wp.shape[0]
    n = 0 if kind == "formula" else (tables[1] if tables else 4096)
    plans = [ops.plan_info(k if n else "exact_" + k, M, K, O, n) for k in ("forward", "backward")]
    ws = [torch.empty(p["contraction_bytes"], dtype=torch.uint8, device=x.device) for p in plans]
    if kind == "formula":
        res = (ops.exact_forward(x, wp, wn, PARAMS, V_SAT, workspace=ws[0]),
               *ops.exact_backward(x, wp, wn, g, PARAMS, V_SAT, True, True, workspace=ws[1]))
        cells = _formula_cells
    else:
        (fwd, bwd), n, lo, hi, cells = tables or _tables(flash_cfg(4096))
        res = (ops.lut_forward(x, wp, wn, fwd, n, lo, hi, V_SAT, -1e30, 1e30, workspace=ws[0]),
               *ops.lut_backward(x, wp, wn, g, bwd, n, lo, hi, V_SAT, True, True, workspace=ws[1]))
    torch.cuda.synchronize()
    if took is not None:
        assert [ops.took_contraction(w, p) for w, p in zip(ws, plans)] == list(took)
    return res, cells


def _inputs(kind, seed, spread=SPREAD):
    M, K, O = SHAPE[kind]
    gen = torch.Generator().manual_seed(seed)
    wp, wn = (2.5 + spread * (torch.rand(O, K, generator=gen) - 0.5) for _ in range(2))
    x = torch.rand(M, K, generator=gen)  # to be placed
    return [t.cuda() for t in (x, wp, wn, torch.randn(M, O, generator=gen))]


def _check(what, got, ref, scale, dims, tol, where=None):
    """The largest error of a group (a row: dims 1, a column: 0) against the group's scale."""
    e, s = (got.double() - ref), scale
    if where is not None:
        e, s = e[where], s[where]
    worst = float((e.norm(dim=dims) / s.norm(dim=dims)).max())
    print(f"  {what}: {worst:.2e}", flush=True)
    assert worst <= tol, (what, worst)


@pytest.mark.parametrize("kind", ["formula", "table"])
@pytest.mark.parametrize("low", [-1.0, 0.2, 0.9])
def test_tokens_without_gradient(cuda_device, kind, low):
    """Half the tokens lie at 3 to 4 V and carry no gradient (padding, or outputs that the layer clamps):
    dVth comes from the others alone, whose slopes are 1e-2 to 1e-16 of theirs."""
    x, wp, wn, g = _inputs(kind, 1)
    x = torch.where((torch.arange(x.shape[0], device="cuda") % 2 == 0)[:, None], low + 0.4 * x, 3.0 + x)
    g[1::2] = 0.0
    print(f"[case] {kind}, tokens without a gradient, the others at {low} V", flush=True)
    got, cells = _run(kind, x, wp, wn, g)
    ref, scale = _reference(x, wp, wn, g, cells)
    for i, name in ((2, "dVth+"), (3, "dVth-")):
        _check(f"{name} by input", got[i], ref[i], scale[i], 0, TOL[kind])
        _check(f"{name} by output", got[i], ref[i], scale[i], 1, TOL[kind])


@pytest.mark.parametrize("kind", ["formula", "table"])
def test_outputs_without_gradient(cuda_device, kind):
    """The high tokens' gradients are masked output by output."""
    x, wp, wn, g = _inputs(kind, 2)
    high = (torch.arange(x.shape[0], device="cuda") % 2 == 1)
    x = torch.where(high[:, None], 3.0 + x, 0.3 + 0.4 * x)
    gen = torch.Generator(device="cuda").manual_seed(3)
    masked = torch.rand(wp.shape[0], device="cuda", generator=gen) < 0.5
    g[high[:, None] & masked[None]] = 0.0
    print(f"[case] {kind}, outputs without a gradient", flush=True)
    got, cells = _run(kind, x, wp, wn, g)
    ref, scale = _reference(x, wp, wn, g, cells)
    for i, name in ((2, "dVth+"), (3, "dVth-")):
        _check(f"{name} of masked outputs", got[i], ref[i], scale[i], 1, TOL[kind], masked)
        _check(f"{name} of the others", got[i], ref[i], scale[i], 1, TOL[kind], ~masked)


@pytest.mark.parametrize("kind", ["formula", "table"])
@pytest.mark.parametrize("low", [-1.0, 0.2])
def test_high_inputs_with_equal_thresholds(cuda_device, kind, low):
    """Inputs at 3 to 4 V whose two thresholds are equal add nothing: the outputs are the other inputs'."""
    x, wp, wn, g = _inputs(kind, 4)
    x[:, 8:] = low + 0.4 * x[:, 8:]
    x[:, :8] += 3.0
    wn[:, :8] = wp[:, :8]
    print(f"[case] {kind}, equal thresholds at the high inputs, the others at {low} V", flush=True)
    got, cells = _run(kind, x, wp, wn, g)
    ref, scale = _reference(x, wp, wn, g, cells)
    _check("out by token", got[0], ref[0], scale[0], 1, TOL[kind])
    _check("out by output", got[0], ref[0], scale[0], 0, TOL[kind])
    _check("dX of the low inputs", got[1][:, 8:], ref[1][:, 8:], scale[1][:, 8:], 1, TOL[kind])
    assert float(got[1][:, :8].abs().max()) == 0.0


@pytest.mark.parametrize("kind", ["formula", "table"])
def test_large_gradients_of_outputs_with_equal_thresholds(cuda_device, kind):
    """Outputs whose branches cancel for every input carry gradients 1e6 times the others'."""
    x, wp, wn, g = _inputs(kind, 5)
    x = 4.0 * x - 1.0
    wn[::2] = wp[::2]
    g[:, ::2] *= 1e6
    print(f"[case] {kind}, large gradients of outputs with equal thresholds", flush=True)
    got, cells = _run(kind, x, wp, wn, g)
    ref, scale = _reference(x, wp, wn, g, cells)
    _check("dX by token", got[1], ref[1], scale[1], 1, TOL[kind])
    _check("dX by input", got[1], ref[1], scale[1], 0, TOL[kind])
    # (each branch's own gradient does not cancel)
    _check("dVth+ of the others", got[2], ref[2], scale[2], 1, TOL[kind], slice(1, None, 2))


@pytest.mark.parametrize("kind,entries,spread", [("formula", 0, SPREAD), ("formula", 0, 0.3), ("table", 4096, SPREAD),
                                                 ("table", 4096, 0.3), ("table", 4096, 1.0), ("table", 8192, SPREAD),
                                                 ("table", 8192, 1.0), ("table", 16384, 1.0)])
def test_tokens_of_all_magnitudes(cuda_device, kind, entries, spread):
    """Tokens from -2 to 4 V, and gradients from 1 to 1e-12, token by token; 8 and 16 terms."""
    x, wp, wn, g = _inputs(kind, 6, spread)
    gen = torch.Generator().manual_seed(7)
    M = x.shape[0]
    x = x * 0.3 + (6.0 * torch.rand(M, 1, generator=gen) - 2.0).cuda()
    g = g * torch.exp(-27.6 * torch.rand(M, 1, generator=gen)).cuda()
    print(f"[case] {kind} {entries} over {spread} V, tokens of all magnitudes", flush=True)
    got, cells = _run(kind, x, wp, wn, g, _tables(flash_cfg(entries)) if entries else None,
                      (True, kind == "formula" or spread <= 0.24 or entries >= 6000))
    ref, scale = _reference(x, wp, wn, g, cells)
    _check("out by token", got[0], ref[0], scale[0], 1, TOL[kind])
    _check("dX by token", got[1], ref[1], scale[1], 1, TOL[kind])
    for i, name in ((2, "dVth+"), (3, "dVth-")):
        _check(f"{name} by input", got[i], ref[i], scale[i], 0, TOL[kind])


def _shape_table(shape, n=4096, lo=-9.0, hi=4.0):
    """A smooth table that is not the transistor's, with its slope, as oracle-style float32 arrays."""
    v = torch.linspace(lo, hi, n, dtype=torch.float64)
    if shape == "saturating":
        s = torch.sigmoid(v / 0.13)
        return 1e-6 * s, 1e-6 * s * (1.0 - s) / 0.13
    if shape == "bump":
        s = torch.exp(-0.5 * ((v + 0.6) / 0.9).square())
        return 1e-6 * s, -1e-6 * s * (v + 0.6) / 0.81
    if shape == "falling":
        s = torch.sigmoid(-v / 0.13)
        return 1e-6 * s, -1e-6 * s * (1.0 - s) / 0.13
    if shape == "steep fall":  # rises by 0.1% from entry to entry, falls by 4%
        s = torch.sigmoid(-(v + 0.5) / 0.08)
        f = 1e-6 * torch.exp(0.3 * v) * s
        return f, f * (0.3 - (1.0 - s) / 0.08)
    return 1e-6 * torch.exp(v / 0.4), 2.5e-6 * torch.exp(v / 0.4)  # "exponential"


@pytest.mark.parametrize("shape", ["saturating", "bump", "falling", "steep fall", "exponential"])
def test_tables_of_other_shapes(cuda_device, shape):
    """Packed tables may hold any curve: slopes that fall again, currents that fall, that only grow."""
    from isa.kernels.transformer_ffn import _hip, ops

    lo, hi, n = -9.0, 4.0, 4096
    ti, td = (t.float() for t in _shape_table(shape, n, lo, hi))
    packed = [ops.pack_tables(ti.cuda(), td.cuda(), layout) for layout in (_hip.LUT_FWD, _hip.LUT_BWD)]
    x, wp, wn, g = _inputs("table", 8, 0.05 if shape == "steep fall" else SPREAD)
    x = 3.3 * x  # (further up the saturating curve's differences are its entries' rounding)
    print(f"[case] {shape} table", flush=True)
    got, cells = _run("table", x, wp, wn, g, (packed, n, lo, hi, _table_cells(ti, td, lo, hi)), None)
    ref, scale = _reference(x, wp, wn, g, cells)
    # the table's own fp32 entries round to 6e-8 of the current, the branches' differences are down to
    # 1e-3 of it where a curve is flat
    for i, name in ((0, "out"), (1, "dX"), (2, "dVth+"), (3, "dVth-")):
        _check(f"{name} by row", got[i], ref[i], scale[i], 1, 4e-5)
        _check(f"{name} by column", got[i], ref[i], scale[i], 0, 4e-5)


@pytest.mark.parametrize("entries", [3600, 4000, 4096, 8192])
def test_close_pairs_are_no_further_off_than_per_cell(cuda_device, entries):
    """Thresholds in pairs within 2 mV, inputs far below threshold: a cell's difference is a few
    thousandths of a lookup, and the kinks count most. The median row's error (noise of 3% over these
    sums) against the per-cell kernels' on the same operands."""
    from isa.kernels.transformer_ffn import ops

    M, K, O = 2048, 384, 1536
    gen = torch.Generator(device="cuda").manual_seed(9)
    x, wp, d, g = (torch.rand(*s, generator=gen, device="cuda") for s in ((M, K), (O, K), (O, K), (M, O)))
    x, wp, g = 1.5 * x - 1.0, 2.5 + SPREAD * (wp - 0.5), g - 0.5
    wn = wp + 0.02 * SPREAD * (d - 0.5)
    tables = _tables(flash_cfg(entries))
    got, cells = _run("table", x, wp, wn, g, tables, None)
    (fwd, bwd), n, lo, hi, _ = tables
    ws = [torch.empty(ops.plan_info(k, M, K, O, n)["cell_bytes"], dtype=torch.uint8, device="cuda")
          for k in ("forward", "backward")]
    cell = (ops.lut_forward(x, wp, wn, fwd, n, lo, hi, V_SAT, -1e30, 1e30, workspace=ws[0]),
            ops.lut_backward(x, wp, wn, g, bwd, n, lo, hi, V_SAT, True, True, workspace=ws[1])[0])
    ref, scale = _reference(x, wp, wn, g, cells)
    print(f"[case] {entries} entries, close pairs", flush=True)
    for i, name in ((0, "out"), (1, "dX")):
        e = [float(((t.double() - ref[i]).norm(dim=1) / scale[i].norm(dim=1)).median()) for t in (got[i], cell[i])]
        print(f"  {name}: {e[0]:.2e}, per-cell {e[1]:.2e}", flush=True)
        assert e[0] <= 1.1 * e[1], (name, e)
