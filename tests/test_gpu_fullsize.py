"""Headline-size parity (Physical GPT-L FFN, M = 8 x 1024 tokens, 768 -> 3072 -> 768).

The oracle cannot redo 3.9e10 cell-evals in test time, so each full-size launch is checked
on samples that are exact sub-problems: forward rows and dX rows depend only on their own
token, dVth columns only on their own output (summed over all 8192 tokens). Size-independent
properties (bitwise determinism, the equal-threshold invariant) run on the full tensors.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.helpers import errs, flash_cfg, make_inputs

pytestmark = pytest.mark.gpu


def _run(x, vp, vn, g, cfg, dev, modes=None, cells=True):
    """Forward and backward through the C ABI, by the per-cell kernels (a workspace of their plan) or,
    cells False, with the workspace in which the matrix cores may take the calls; modes (a dict)
    receives the table mode each main kernel ran in (1 two copies, 0 one copy, 2 the ranked
    backward, 64 the matrix cores, None no second copy in the plan)."""
    from isa.approximations.delta_lut import get_packed_tables, lut_range
    from isa.kernels.transformer_ffn import ops

    dmin, dmax, n = lut_range(cfg)
    fwd, bwd = get_packed_tables(cfg, dev)
    M, K = x.shape
    O = vp.shape[0]
    pf, pb = ops.plan_info("forward", M, K, O, n), ops.plan_info("backward", M, K, O, n)
    size = "cell_bytes" if cells else "contraction_bytes"
    wsf, wsb = (torch.empty(p[size], dtype=torch.uint8, device=dev) for p in (pf, pb))
    out = ops.lut_forward(x, vp, vn, fwd, n, dmin, dmax, cfg["V_sat"], -4.0, 4.0, workspace=wsf)
    gx, gp, gn = ops.lut_backward(x, vp, vn, g, bwd, n, dmin, dmax, cfg["V_sat"], True, True, workspace=wsb)
    torch.cuda.synchronize()
    if modes is not None:
        modes["fwd"], modes["bwd"] = ops.copy_mode(wsf, pf), ops.copy_mode(wsb, pb)
    return out, gx, gp, gn


def _check_samples(x, vp, vn, g, res, cfg, rng, n_rows=48, n_cols=24):
    out, gx, gp, gn = res
    dmin, dmax, n = oracle.lut_range(cfg)
    ti, td = oracle.lut_tables(cfg)
    X, P, N, G = (t.cpu().numpy() for t in (x, vp, vn, g))
    rows = np.sort(rng.choice(X.shape[0], n_rows, replace=False))
    cols = np.sort(rng.choice(P.shape[0], n_cols, replace=False))
    ref = oracle.forward(X[rows], P, N, ti, dmin, dmax, cfg["V_sat"])
    rdx = oracle.grad_x(X[rows], P, N, G[rows], ti, td, dmin, dmax, cfg["V_sat"])
    rgp, rgn = oracle.grad_w(X, P[cols], N[cols], np.ascontiguousarray(G[:, cols]), td, dmin, dmax, cfg["V_sat"])
    e = {"fwd": errs(out[rows], ref), "dX": errs(gx[rows], rdx),
         "dVth+": errs(gp[cols], rgp), "dVth-": errs(gn[cols], rgn)}
    print({k: f"{v[0]:.2e}/{v[1]:.2e}" for k, v in e.items()})
    assert e["fwd"][0] <= 1e-4
    assert max(e["dX"][0], e["dVth+"][0], e["dVth-"][0]) <= 1e-3


def test_headline_ffn_layers_on_the_matrix_cores(cuda_device):
    """What the headline runs at its initial thresholds, both layers, forward and backward."""
    from isa.kernels.transformer_ffn import ops

    print("[case] headline fc1, fc2 on the matrix cores, M=8192", flush=True)
    cfg = flash_cfg(4096)
    rng = np.random.default_rng(0)
    x, vp, vn, g = (t.to(cuda_device) for t in make_inputs(8192, 768, 3072, seed=0))
    for _ in range(2):
        modes = {}
        res = _run(x, vp, vn, g, cfg, cuda_device, modes, cells=False)
        assert modes["fwd"] == modes["bwd"] == ops.MODE_CONTRACTION, modes
        _check_samples(x, vp, vn, g, res, cfg, rng)
        for a, b in zip(res, _run(x, vp, vn, g, cfg, cuda_device, cells=False)):
            assert torch.equal(a, b)
        x = (res[0] * 1e5).clamp(-4.0, 4.0).contiguous()  # fc2's inputs
        _, vp, vn, _ = (t.to(cuda_device) for t in make_inputs(1, 3072, 768, seed=1))
        g = torch.randn(8192, 768, generator=torch.Generator().manual_seed(2)).to(cuda_device)


def test_headline_ffn_layers(cuda_device):
    print("[case] headline fc1 768->3072, fc2 3072->768, M=8192", flush=True)
    cfg = flash_cfg(4096)
    rng = np.random.default_rng(0)
    x, vp, vn, g = (t.to(cuda_device) for t in make_inputs(8192, 768, 3072, seed=0))
    modes = {}
    res1 = _run(x, vp, vn, g, cfg, cuda_device, modes)
    # the initial thresholds span ~69 records and the mapped inputs ~1350: the forward holds as
    # many windowed table copies as fit its 80 KB of LDS (about seven); the backward runs ranked
    assert 3 <= modes["fwd"] <= 32 and modes["bwd"] == 2, modes
    _check_samples(x, vp, vn, g, res1, cfg, rng)
    # fc2 is driven by the TIA output of fc1: clamp(R_TIA * Idiff, -4, 4) (cim.py:192-193)
    x2 = (res1[0] * 1e5).clamp(-4.0, 4.0).contiguous()
    frac_sat = float((x2.abs() >= 4.0).float().mean())
    print(f"fc2 input saturation {frac_sat:.3f}")
    _, vp2, vn2, g2 = make_inputs(1, 3072, 768, seed=1)
    g2 = torch.randn(8192, 768, generator=torch.Generator().manual_seed(2))
    vp2, vn2, g2 = (t.to(cuda_device) for t in (vp2, vn2, g2))
    res2 = _run(x2, vp2, vn2, g2, cfg, cuda_device)
    _check_samples(x2, vp2, vn2, g2, res2, cfg, rng)
    # bitwise determinism at full size
    again = _run(x2, vp2, vn2, g2, cfg, cuda_device)
    for a, b in zip(res2, again):
        assert torch.equal(a, b)


def test_headline_equal_threshold_invariant(cuda_device):
    """vth_pos == vth_neg: exactly zero Idiff, dVth+ == -dVth- bitwise, and dX zero to rounding
    (the ranked backward, which runs here, sums an output's + and - branches in separate slots:
    bounded by 1e-6 of the dX magnitude of the same inputs with distinct thresholds)."""
    cfg = flash_cfg(4096)
    x, vp, vn, g = (t.to(cuda_device) for t in make_inputs(8192, 768, 3072, seed=5))
    modes = {}
    out, gx, gp, gn = _run(x, vp, vp, g, cfg, cuda_device, modes)
    assert modes["bwd"] == 2, modes
    assert torch.count_nonzero(out) == 0
    assert torch.equal(gp, -gn)
    scale = float(_run(x, vp, vn, g, cfg, cuda_device)[1].abs().max())
    print(f"max |dX| {float(gx.abs().max()):.3e} of dX scale {scale:.3e}")
    assert float(gx.abs().max()) <= 1e-6 * scale


@pytest.mark.parametrize("size,vth_mode", [(8192, "init"), (4096, "full"), (16384, "init")])
def test_headline_fc1_table_copies(cuda_device, size, vth_mode):
    """The regimes where the kernels hold a second, bank-rotated table copy, at the headline
    fc1 shape: the 8192-entry table (its initial thresholds span ~135 records; the forward
    runs its table copies in one 16-wave block per CU, each wave summing all 768 inputs) and
    thresholds spread over U[V_TH_MIN, V_TH_MAX] (forward copies, and the persistent
    two-copy backward); and the 16384-entry table (one 131 KB copy per CU in the forward, the
    backward from global memory), checked on sampled exact sub-problems."""
    print(f"[case] headline fc1 with table copies: {size} entries, thresholds {vth_mode}", flush=True)
    cfg = flash_cfg(size)
    rng = np.random.default_rng(size)
    x, vp, vn, g = (t.to(cuda_device) for t in make_inputs(8192, 768, 3072, seed=7, vth_mode=vth_mode))
    modes = {}
    res = _run(x, vp, vn, g, cfg, cuda_device, modes)
    # 16384 entries: no LDS room for a second full copy; the forward holds three windowed copies
    # in its one-copy allocation when its window is short enough, the backward reads the table
    # from global memory (no mode). 8192 entries at the initial thresholds: the forward holds
    # windowed copies in its 16-wave blocks, the backward runs ranked (135 records). The wide
    # spread: windowed forward copies of a ~2900-record window (three fit), the two-copy
    # backward (1576 records, past the ranked kernel's 420), with windowed copies where they fit
    if size > 8192:
        assert modes["bwd"] is None and (modes["fwd"] in (0, 33) or 3 <= modes["fwd"] <= 32), modes
    else:
        if vth_mode == "init":
            assert 3 <= modes["fwd"] <= 32 and modes["bwd"] == 2, modes
        else:  # the two-copy launch, with windowed copies (33: two) where the window fits
            assert (3 <= modes["fwd"] <= 32 or modes["fwd"] == 33) and (modes["bwd"] in (1, 33) or
                                                                      3 <= modes["bwd"] <= 32), modes
    _check_samples(x, vp, vn, g, res, cfg, rng)
    again = _run(x, vp, vn, g, cfg, cuda_device)
    for a, b in zip(res, again):
        assert torch.equal(a, b)
