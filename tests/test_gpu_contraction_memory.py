"""GPU test of calls whose workspace does not fit the device with the matrix cores' operands: they run
the per-cell kernels in a workspace of their plan, with those kernels' bits."""

from __future__ import annotations

import pytest
import torch

from tests.helpers import flash_cfg
from tests.test_gpu_contraction import PARAMS, V_SAT

pytestmark = pytest.mark.gpu

M, K, O, N = 2048, 384, 1536, 4096


def _calls():
    """name -> (plan_info arguments, the call with keyword arguments to pass on)."""
    from isa.approximations.delta_lut import get_packed_tables, lut_range
    from isa.kernels.transformer_ffn import ops

    cfg = flash_cfg(N)
    lo, hi, n = lut_range(cfg)
    fwd, bwd = get_packed_tables(cfg, torch.device("cuda"))
    g = torch.Generator().manual_seed(0)
    x = (torch.rand(M, K, generator=g) * 4.0).cuda()
    wp, wn = ((2.5 + 0.2142 * (torch.rand(O, K, generator=g) - 0.5)).cuda() for _ in range(2))
    grad, gain = torch.randn(M, O, generator=g).cuda(), torch.tensor([0.2], device="cuda")
    out = (-1e30, 1e30)

    def layer_forward(**kw):
        return ops.lut_layer_forward(x, wp, wn, fwd, n, lo, hi, V_SAT, *out, r_tia=gain, y_range=out, **kw)

    def layer_backward(**kw):
        r = ops.lut_layer_backward(x, wp, wn, grad, idiff, bwd, n, lo, hi, V_SAT, need_grad_x=True, need_grad_w=True,
                                   r_tia=gain, y_range=out, **kw)
        return r["dx"], r["dvth_pos"], r["dvth_neg"]

    idiff = layer_forward()[1]
    shape = (M, K, O)
    return {
        "forward": (("forward", *shape, n), lambda **kw: [ops.lut_forward(x, wp, wn, fwd, n, lo, hi, V_SAT, *out, **kw)]),
        "backward": (("backward", *shape, n),
                     lambda **kw: ops.lut_backward(x, wp, wn, grad, bwd, n, lo, hi, V_SAT, True, True, **kw)),
        "layer_forward": (("forward", *shape, n), layer_forward),
        "layer_backward": (("layer_backward", *shape, n), layer_backward),
        "exact_forward": (("exact_forward", *shape, 0), lambda **kw: [ops.exact_forward(x, wp, wn, PARAMS, V_SAT, **kw)]),
        "exact_backward": (("exact_backward", *shape, 0),
                           lambda **kw: ops.exact_backward(x, wp, wn, grad, PARAMS, V_SAT, True, True, **kw)),
    }


@pytest.mark.parametrize("name", ["forward", "backward", "layer_forward", "layer_backward", "exact_forward",
                                  "exact_backward"])
def test_call_without_room_for_its_operands(cuda_device, monkeypatch, name):
    from isa.kernels.transformer_ffn import ops

    plan_args, call = _calls()[name]
    plan = ops.plan_info(*plan_args)
    cells = torch.empty(plan["cell_bytes"], dtype=torch.uint8, device="cuda")
    want = [t.clone() for t in call(workspace=cells)]
    full = torch.empty(plan["contraction_bytes"], dtype=torch.uint8, device="cuda")
    taken = call(workspace=full)
    torch.cuda.synchronize()
    assert ops.took_contraction(full, plan) and not torch.equal(taken[0], want[0])
    empty, sizes = torch.empty, []

    def limited(*size, **kw):
        if kw.get("dtype") is torch.uint8:
            sizes.append(size[0])
            if size[0] > plan["cell_bytes"]:
                raise torch.OutOfMemoryError("no room")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", limited)
    got = call()
    torch.cuda.synchronize()
    monkeypatch.undo()
    assert sizes == [plan["contraction_bytes"], plan["cell_bytes"]]
    for a, b in zip(got, want):
        assert torch.equal(a, b)

    def none(*size, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", none)
    with pytest.raises(torch.OutOfMemoryError):
        call()


@pytest.mark.parametrize("kind,tokens", [("forward", 21500), ("backward", 29000)])
def test_operands_past_2_gib(cuda_device, kind, tokens):
    """3072 -> 768 with as many tokens as the operands' limits take: offsets of up to 4 GiB. The first and
    last tokens (and dVth, a sum over all of them) against the per-cell kernels: 1.5e-5 is what the two
    paths' roundings (1e-5 and 4e-6) add up to."""
    from isa.approximations.delta_lut import get_packed_tables, lut_range
    from isa.kernels.transformer_ffn import ops

    k, o = 3072, 768
    cfg = flash_cfg(N)
    lo, hi, n = lut_range(cfg)
    fwd, bwd = get_packed_tables(cfg, torch.device("cuda"))
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand(tokens, k, generator=gen, device="cuda") * 4.0
    wp, wn = (2.5 + 0.2142 * (torch.rand(o, k, generator=gen, device="cuda") - 0.5) for _ in range(2))
    plan = ops.plan_info(kind, tokens, k, o, n)
    assert plan["contraction_bytes"] - plan["cell_bytes"] > 4 << 30
    print(f"[case] {kind} {tokens} x {k} -> {o}, {plan['contraction_bytes'] / 1e9:.1f} GB", flush=True)
    if kind == "forward":
        def call(ws):
            return [ops.lut_forward(x, wp, wn, fwd, n, lo, hi, V_SAT, -1e30, 1e30, workspace=ws)]
    else:
        grad = torch.randn(tokens, o, generator=gen, device="cuda")

        def call(ws):
            return ops.lut_backward(x, wp, wn, grad, bwd, n, lo, hi, V_SAT, True, True, workspace=ws)

    ws = torch.empty(plan["contraction_bytes"], dtype=torch.uint8, device="cuda")
    got = call(ws)
    torch.cuda.synchronize()
    assert ops.took_contraction(ws, plan)
    want = call(ws[:plan["cell_bytes"]])
    for a, b in zip(got, want):
        for rows in (slice(0, 300), slice(-300, None)):
            e = float((a[rows] - b[rows]).norm() / b[rows].norm())
            print(f"  {e:.2e}", flush=True)
            assert e <= 1.5e-5, e
