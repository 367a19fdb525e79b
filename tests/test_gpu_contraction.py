"""GPU tests of the projection as a contraction on the matrix cores (contraction.hpp), against
the formula and its analytic gradients in float64 (oracle/exact.py, evaluated on the device in
chunks of rows).

Tolerance: the operands carry 2^-24 of each value, pairs, singles and the truncated series 3e-7; a
sum over n inner elements is taken in slabs of 16, added in fp32 to about sqrt(n / 32) * 2^-24 of its
largest partial sum: 1.7e-6 at the largest sums here (n = 2 terms x 5800 inputs), norm-wise. The
per-cell kernels' own gate is 1e-4; which of the two ran is asserted in every test.
"""

from __future__ import annotations

import pytest
import torch

from oracle import exact
from tests.helpers import flash_cfg

pytestmark = pytest.mark.gpu

TOL = 2e-6
PARAMS = (4.1360, 0.0259, 7.5875e-7, 0.1)
V_SAT = 8.2624


def _inputs(M, K, O, spread, seed=0, x_lo=0.0, x_hi=4.0):
    g = torch.Generator().manual_seed(seed)
    x = torch.rand(M, K, generator=g) * (x_hi - x_lo) + x_lo
    wp, wn = (2.5 + spread * (torch.rand(O, K, generator=g) - 0.5) for _ in range(2))
    # rows of G over four orders of magnitude, as tokens' gradients are
    grad = torch.randn(M, O, generator=g) * torch.exp(-9.0 * torch.rand(M, 1, generator=g))
    return [t.cuda() for t in (x, wp, wn, grad)]


def _reference(x, wp, wn, g):
    cfg = flash_cfg(4096, ekv_approx="exact")
    xd, pd, nd, gd = (t.double() for t in (x, wp, wn, g))
    step = max(1, int(2e7 // max(1, wp.numel())))
    out, dx, dp, dn = [], [], torch.zeros_like(pd), torch.zeros_like(nd)
    for a in range(0, x.shape[0], step):
        b = slice(a, a + step)
        out.append(exact.diff_current_f64(xd[b], pd, nd, cfg))
        gx, gp, gn = exact.diff_current_grads_f64(xd[b], pd, nd, gd[b], cfg)
        dx.append(gx)
        dp += gp
        dn += gn
    return torch.cat(out), torch.cat(dx), dp, dn


def _run(x, wp, wn, g, need_x=True, need_w=True, took=None):
    """took: whether the contraction has to have taken both calls, or to have refused them."""
    from isa.kernels.transformer_ffn import ops

    (M, K), O = x.shape, wp.shape[0]
    plans = [ops.plan_info(k, M, K, O, 0, need_x, need_w) for k in ("exact_forward", "exact_backward")]
    ws = [torch.empty(p["contraction_bytes"], dtype=torch.uint8, device=x.device) for p in plans]
    out = ops.exact_forward(x, wp, wn, PARAMS, V_SAT, workspace=ws[0])
    res = (out, *ops.exact_backward(x, wp, wn, g, PARAMS, V_SAT, need_x, need_w, workspace=ws[1]))
    torch.cuda.synchronize()
    if took is not None:
        assert [ops.took_contraction(w, p) for w, p in zip(ws, plans)] == [took, took]
    return res


def _errors(got, ref):
    return [float((a.double() - r).abs().max() / r.abs().max()) for a, r in zip(got, ref)]


# (M, K, O, threshold spread in volts): from 2^29 cells 8 terms up to 0.24 V, 16 to 0.31 V, then the
# per-cell kernels; remainders of the 128 and 256 tiles, of the 32-element slabs and of the inputs'
# fours; few tokens, few inputs, few outputs
CASES = [
    (3700, 192, 768, 0.2142),
    (16, 5800, 5801, 0.2142),
    (1757, 515, 600, 0.2142),
    (29001, 9, 2100, 0.2142),
    (58001, 500, 19, 0.2142),
    (1361, 770, 513, 0.2142),
    (4201, 389, 333, 0.3),
    (15501, 67, 523, 0.31),
    (1341, 390, 1027, 0.28),
    (2048, 700, 1031, 4.9),
]


@pytest.mark.parametrize("M,K,O,spread", CASES)
def test_contraction_matches_formula(cuda_device, M, K, O, spread):
    print(f"[case] contraction M={M} K={K} O={O} spread={spread}", flush=True)
    x, wp, wn, g = _inputs(M, K, O, spread, seed=M + K, x_lo=-3.0)
    got = _run(x, wp, wn, g, took=spread <= 0.31)
    e = _errors(got, _reference(x, wp, wn, g))
    print(["%.2e" % v for v in e], flush=True)
    assert max(e) <= (TOL if spread <= 0.31 else 6e-6), e
    for a, b in zip(got, _run(x, wp, wn, g)):
        assert torch.equal(a, b)


def test_contraction_rows_keep_their_precision(cuda_device):
    """A token far below threshold beside others far above: its outputs are 1e-9 of theirs, and
    so are its gradients; each is compared against its own scale."""
    x, wp, wn, g = _inputs(3700, 192, 768, 0.2142, seed=3)
    x[::2] = x[::2] * 0.1 - 1.5
    got, ref = _run(x, wp, wn, g, took=True), _reference(x, wp, wn, g)
    for a, r in zip(got[:2], ref[:2]):  # (dVth, a sum over the tokens: test_gpu_contraction_scales.py)
        e = (a.double() - r).abs().amax(1) / r.abs().amax(1)
        assert float(e.max()) <= TOL, float(e.max())


def test_contraction_invariants(cuda_device):
    x, wp, wn, g = _inputs(3700, 192, 768, 0.2142, seed=5)
    out, gx, gp, gn = _run(x, wp, wp, g, took=True)
    assert float(out.abs().max()) == 0.0 and float(gx.abs().max()) == 0.0 and torch.equal(gp, -gn)
    # swapped thresholds negate every operand; the matrix cores' sums of 16 products do not
    # round symmetrically about zero, so the outputs agree to the sums' rounding
    a, b = _run(x, wp, wn, g)[0], -_run(x, wn, wp, g)[0]
    assert float((a - b).abs().max() / a.abs().max()) <= TOL
    full, only_x, only_w = (_run(x, wp, wn, g, *need, took=True) for need in ((True, True), (True, False), (False, True)))
    assert torch.equal(full[1], only_x[1]) and torch.equal(full[2], only_w[2]) and torch.equal(full[3], only_w[3])


@pytest.mark.parametrize("what", ["spread", "range", "nan", "inf", "negative"])
def test_calls_that_do_not_suit(cuda_device, what):
    """Operands that the contraction does not take run the per-cell kernels in the same call:
    thresholds spread too far, x near -V_sat or over more than the table holds, non-finite
    values (whose rows alone are non-finite)."""
    x, wp, wn, g = _inputs(3700, 192, 768, 6.0 if what == "spread" else 0.2142, seed=7)
    bad = None
    if what == "range":
        x[5, 7] = 39.0
    elif what == "negative":
        x[5, 7] = -7.9
    elif what == "nan":
        x[5, 7] = float("nan")
        bad = 5
    elif what == "inf":
        g[9, 3] = float("inf")
    out, gx, gp, gn = _run(x, wp, wn, g, took=None if what == "inf" else False)
    if what == "inf":  # (G's: the forward is taken)
        assert torch.isfinite(out).all() and not torch.isfinite(gx[9]).any()
        keep = torch.arange(3700, device="cuda") != 9
        assert torch.isfinite(gx[keep]).all()
        assert not torch.isfinite(gp[3]).any() and torch.isfinite(gp[4]).all()
        return
    if bad is not None:
        assert torch.isnan(out[bad]).all()
        keep = torch.arange(3700, device="cuda") != bad
        assert torch.isfinite(out[keep]).all()
        return
    e = _errors((out, gx, gp, gn), _reference(x, wp, wn, g))
    assert max(e) <= 1e-4, e


def test_contraction_replays_from_a_graph(cuda_device):
    """A captured forward and backward, replayed with thresholds that change the number of terms
    and the path between the replays, equals the eager calls bitwise."""
    from isa.kernels.transformer_ffn import ops

    x, wp, wn, g = _inputs(3700, 192, 768, 0.2142, seed=9)
    static = [t.clone() for t in (x, wp, wn, g)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _run(*static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.exact_forward(*static[:3], PARAMS, V_SAT)
        grads = ops.exact_backward(*static, PARAMS, V_SAT, True, True)
    for spread in (0.2142, 0.3, 6.0, 0.2142):
        x, wp, wn, g = _inputs(3700, 192, 768, spread, seed=int(spread * 100))
        for s, t in zip(static, (x, wp, wn, g)):
            s.copy_(t)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip((out, *grads), _run(x, wp, wn, g)):
            assert torch.equal(a, b), spread
