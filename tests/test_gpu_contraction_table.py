"""GPU tests of the table projection as a contraction on the matrix cores (contraction.hpp),
against lookups in the oracle's table in float64, on the device in chunks of rows.

Tolerance (2-norm): four harmonics leave S / (2 pi^2) sum_(q > 4) cos(2 pi q c) / q^2 of a lookup's
kinks, root mean square 0.0021 S, with S = growth^2 of the entry (growth 3% from entry to entry below
threshold at 4096 entries, as 1 / entries), and fewer where growth allows: 4e-6 of the branches'
difference there, whose rms is 27 entries' growth. What the two functions of the threshold leave is as
much again for dX around 3 V (5e-6 for the slopes), less elsewhere. The outputs' norms are those of the
inputs well above threshold, where the kinks are smaller: half of the sum, 5e-6, is allowed. The
per-cell kernels' own gate is 1e-4; which of the two ran is asserted in every test.
"""

from __future__ import annotations

import pytest
import torch

from tests.helpers import flash_cfg, oracle_tables

pytestmark = pytest.mark.gpu

V_SAT = 8.2624


TOL = 5e-6
CELL_TOL = 2e-5  # the per-cell kernels, 2-norm


def _inputs(M, K, O, spread, seed=0, x_lo=-4.0, x_hi=4.0):
    g = torch.Generator().manual_seed(seed)
    x = torch.rand(M, K, generator=g) * (x_hi - x_lo) + x_lo
    wp, wn = (2.5 + spread * (torch.rand(O, K, generator=g) - 0.5) for _ in range(2))
    grad = torch.randn(M, O, generator=g) * torch.exp(-9.0 * torch.rand(M, 1, generator=g))
    return [t.cuda() for t in (x, wp, wn, grad)]


def _reference(x, wp, wn, g, cfg):
    from isa.approximations.delta_lut import lut_range

    lo, hi, n = lut_range(cfg)
    ti, td = (torch.as_tensor(t, dtype=torch.float64).cuda() for t in oracle_tables(cfg))
    xd, wd, gd = x.double(), [w.double() for w in (wp, wn)], g.double()

    def lookup(tables, v):
        c = ((v - lo) * ((n - 1) / (hi - lo))).clamp(0, n - 1)
        i = c.floor().clamp(max=n - 2).long()
        f = c - i
        return [t[i] + f * (t[i + 1] - t[i]) for t in tables]

    r = 1.0 / (1.0 + xd / V_SAT)
    out, dx = torch.zeros_like(gd), torch.zeros_like(xd)
    dw = [torch.zeros_like(w) for w in wd]
    step = max(1, int(1e7 // wp.numel()))
    for a in range(0, x.shape[0], step):
        b = slice(a, a + step)
        for q, sign in ((0, 1.0), (1, -1.0)):
            cur, slope = lookup((ti, td), xd[b, None, :] - wd[q][None])
            out[b] += sign * (cur * r[b, None, :]).sum(2)
            dx[b] += sign * ((slope * r[b, None, :] - cur * r[b, None, :] ** 2 / V_SAT) * gd[b, :, None]).sum(1)
            dw[q] -= sign * (slope * r[b, None, :] * gd[b, :, None]).sum(0)
    return out, dx, dw[0], dw[1]


def _tables(cfg):
    from isa.approximations.delta_lut import get_packed_tables, lut_range

    lo, hi, n = lut_range(cfg)
    fwd, bwd = get_packed_tables(cfg, torch.device("cuda"))
    return fwd, bwd, n, lo, hi


def _run(x, wp, wn, g, cfg, need_x=True, need_w=True, took=None):
    """took: whether the contraction has to have taken the forward and the backward."""
    from isa.kernels.transformer_ffn import ops

    fwd, bwd, n, lo, hi = _tables(cfg)
    (M, K), O = x.shape, wp.shape[0]
    plans = [ops.plan_info(k, M, K, O, n, need_x, need_w) for k in ("forward", "backward")]
    ws = [torch.empty(p["contraction_bytes"], dtype=torch.uint8, device=x.device) for p in plans]
    out = ops.lut_forward(x, wp, wn, fwd, n, lo, hi, V_SAT, -1e30, 1e30, workspace=ws[0])
    res = (out, *ops.lut_backward(x, wp, wn, g, bwd, n, lo, hi, V_SAT, need_x, need_w, workspace=ws[1]))
    torch.cuda.synchronize()
    if took is not None:
        assert [ops.took_contraction(w, p) for w, p in zip(ws, plans)] == list(took)
        for w, p, t in zip(ws, plans, took):
            mode = ops.copy_mode(w, p)
            assert mode is None or (mode == ops.MODE_CONTRACTION) == t, mode
    return res


def _per_cell(x, wp, wn, g, cfg):
    """The per-cell kernels on the same operands: a workspace that only their plan fits."""
    from isa.kernels.transformer_ffn import ops

    M, K, O = x.shape[0], x.shape[1], wp.shape[0]
    fwd, bwd, n, lo, hi = _tables(cfg)
    ws = torch.empty(ops.plan_info("forward", M, K, O, n)["cell_bytes"], dtype=torch.uint8, device="cuda")
    return ops.lut_forward(x, wp, wn, fwd, n, lo, hi, V_SAT, -1e30, 1e30, workspace=ws)


def _errors(got, ref):
    return [float((a.double() - r).norm() / r.norm()) for a, r in zip(got, ref)]


# (M, K, O, entries, threshold spread): 2^30 cells and just above; 8 terms up to 0.24 V, 16 to
# 1.07 V (the backward from 6000 entries on); four harmonics (up to 5500 entries), two (8192),
# one (13000, 16384), none (62000); remainders of the 128 and 256 tiles, of the slabs, of the inputs'
# fours and of the table's 256-entry ranges; odd and even inputs; few tokens, few outputs, few inputs
CASES = [
    (2048, 384, 1536, 4096, 0.2142),
    (2111, 389, 1533, 4096, 0.2142),
    (515, 1031, 2051, 4000, 0.2142),
    (2051, 513, 1031, 4000, 0.8),
    (1999, 515, 1101, 4096, 0.3),
    (700, 770, 2003, 62000, 0.2142),
    (2053, 515, 1031, 5500, 0.2142),
    (2048, 511, 1037, 8192, 0.2142),
    (20, 7330, 7330, 4096, 0.2142),
    (18001, 9, 6650, 4099, 0.2142),
    (11001, 5799, 17, 4096, 0.2142),
    (1999, 515, 1100, 4096, 1.0),
    (2060, 513, 1027, 8192, 0.8),
    (1370, 769, 1025, 13000, 0.2142),
    (1369, 770, 1029, 16384, 1.0),
    (2050, 512, 1026, 16384, 0.2142),
]


@pytest.mark.parametrize("M,K,O,entries,spread", CASES)
def test_contraction_matches_lookups(cuda_device, M, K, O, entries, spread):
    print(f"[case] table contraction M={M} K={K} O={O} {entries} entries spread={spread}", flush=True)
    cfg = flash_cfg(entries)
    x, wp, wn, g = _inputs(M, K, O, spread, seed=M + K)
    took = True, spread <= 0.24 or entries >= 6000
    got = _run(x, wp, wn, g, cfg, took=took)
    e = _errors(got, _reference(x, wp, wn, g, cfg))
    print(["%.2e" % v for v in e], flush=True)
    assert e[0] <= TOL and max(e[1:]) <= (TOL if took[1] else CELL_TOL), e
    for a, b in zip(got, _run(x, wp, wn, g, cfg)):
        assert torch.equal(a, b)


def test_table_contraction_takes_the_call(cuda_device):
    """A workspace of the per-cell plan runs the per-cell kernels: other roundings, the same result."""
    cfg = flash_cfg(4096)
    x, wp, wn, g = _inputs(2048, 384, 1536, 0.2142, seed=1)
    out, *grads = _run(x, wp, wn, g, cfg, took=(True, True))
    cell = _per_cell(x, wp, wn, g, cfg)
    assert not torch.equal(out, cell)
    assert float((out - cell).norm() / cell.norm()) <= 3e-5
    only_x, only_w = (_run(x, wp, wn, g, cfg, *need, took=(True, True)) for need in ((True, False), (False, True)))
    assert torch.equal(grads[0], only_x[1]) and torch.equal(grads[1], only_w[2]) and torch.equal(grads[2], only_w[3])


@pytest.mark.parametrize("what", ["spread", "bf16", "low", "high", "outlier", "nan", "inf", "coarse"])
def test_table_calls_that_do_not_suit(cuda_device, what):
    """What the contraction does not take runs the per-cell kernels, with their bits: thresholds
    spread too far (a sample shows it, or, "outlier", one threshold that no sample holds), tables
    that are not smooth or too coarse, lookups past a table end, non-finite operands."""
    cfg = flash_cfg(2048 if what == "coarse" else 4096, **({"LUT_DTYPE": "bfloat16"} if what == "bf16" else {}))
    x, wp, wn, g = _inputs(2048, 384, 1536, 5.0 if what == "spread" else 0.2142, seed=7)
    if what == "low":
        x[5, 7] = -7.9
    elif what == "high":
        x[5, 7] = 30.0
    elif what == "outlier":
        wn[1000, 7] = 4.5
    elif what == "nan":
        x[5, 7] = float("nan")
    elif what == "inf":
        g[9, 3] = float("inf")
    out, gx, gp, gn = _run(x, wp, wn, g, cfg, took=(what == "inf", False))  # (G's: the forward is taken)
    cell = _per_cell(x, wp, wn, g, cfg)
    if what == "nan":
        assert torch.equal(torch.nan_to_num(out, 7.0), torch.nan_to_num(cell, 7.0)) and not torch.isfinite(gx[5, 7])
        keep = torch.arange(2048, device="cuda") != 5
        assert torch.isfinite(out[keep]).all() and torch.isfinite(gx[keep]).all()
        return
    if what == "inf":
        keep = torch.arange(2048, device="cuda") != 9
        assert torch.isfinite(gx[keep]).all() and not torch.isfinite(gx[9]).any()
        assert torch.isfinite(gp[4]).all() and not torch.isfinite(gp[3]).any()
        return
    assert torch.equal(out, cell)
    e = _errors((out, gx, gp, gn), _reference(x, wp, wn, g, cfg))
    assert max(e) <= 1e-4, e


def test_table_contraction_with_glue(cuda_device):
    """The layer form against the plain one: input mapping, gain, statistics and gradients."""
    from isa.kernels.transformer_ffn import ops

    cfg = flash_cfg(4096)
    M, K, O = 2049, 385, 1537
    x, wp, wn, g = _inputs(M, K, O, 0.2142, seed=3, x_lo=-0.7, x_hi=1.0)
    fwd, bwd, n, lo, hi = _tables(cfg)
    aff = torch.tensor([2.0, 1.5], device="cuda")
    gain = torch.tensor([0.2], device="cuda")
    top, total = torch.zeros(1, device="cuda"), torch.zeros(1, dtype=torch.float64, device="cuda")
    out, idiff = ops.lut_layer_forward(x, wp, wn, fwd, n, lo, hi, V_SAT, -1e30, 1e30, in_affine=aff, r_tia=gain,
                                       y_range=(-1e30, 1e30), stat_abs_max=top, stat_total=total)
    plain = _run(x * 2.0 + 1.5, wp, wn, g * 0.2, cfg)[0]
    assert float((out - plain * 0.2).norm() / out.norm()) <= 1e-6
    assert float(top) == float(out.abs().max()) and float(total) == M * O
    ref = _reference(x * 2.0 + 1.5, wp, wn, g * 0.2, cfg)
    grads = ops.lut_layer_backward(x, wp, wn, g, idiff, bwd, n, lo, hi, V_SAT, need_grad_x=True, need_grad_w=True,
                                   in_affine=aff, r_tia=gain, y_range=(-1e30, 1e30))
    e = _errors((grads["dx"] / 2.0, grads["dvth_pos"], grads["dvth_neg"]), ref[1:])
    assert max(e) <= TOL, e


def test_table_contraction_replays_from_a_graph(cuda_device):
    """A captured forward and backward, replayed with operands that change the number of terms and
    the path between the replays, equals the eager calls bitwise."""
    cfg = flash_cfg(4096)
    static = _inputs(2048, 384, 1536, 0.2142, seed=9)
    _tables(cfg)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _run(*static, cfg)
    torch.cuda.current_stream().wait_stream(side)
    from isa.kernels.transformer_ffn import ops

    fwd, bwd, n, lo, hi = _tables(cfg)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.lut_forward(*static[:3], fwd, n, lo, hi, V_SAT, -1e30, 1e30)
        grads = ops.lut_backward(*static, bwd, n, lo, hi, V_SAT, True, True)
    for spread in (0.2142, 0.8, 5.0, 0.2142):
        for s, t in zip(static, _inputs(2048, 384, 1536, spread, seed=int(spread * 100))):
            s.copy_(t)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip((out, *grads), _run(*static, cfg)):
            assert torch.equal(a, b), spread
