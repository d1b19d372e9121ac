"""The fused GEMMs where their software pipelines begin and end: contractions of one to five 64-wide
steps (the rings hold three or four), the input gradient's partial last step next to values that must
not leak in, the SwiGLU epilogue on tiles of 224 and 256 tokens, and the small-M kernel's last items.
Bounds: the parity bar of assert_close; fused against separate launches of one plan: the same bits."""

import pytest
import torch

from helpers import assert_close, make_weight, oracle_state, randn16
from oracle import nf4 as O

pytestmark = pytest.mark.gpu

ROWS = {2: 64, 4: 128, 7: 224, 8: 256, 9: 288}


@pytest.mark.parametrize("nested", [True, False])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("blocks", [2, 4, 7, 8, 9])
def test_forward_few_steps(blocks, steps, nested, device, monkeypatch):
    from decik_amd.nf4 import launch_plan, linear_forward

    monkeypatch.setenv("DECIK_FWD_PLAN", f"{blocks},1,8")
    m, n, k = ROWS[blocks] + 1, 264, 64 * steps
    plan = launch_plan(False, m, k, [n])
    assert plan["kernel"] == "nf4_fwd8_kernel" and plan["rows_blocks"] == blocks
    packed, qs, w = make_weight((n, k), seed=steps, device=device, nested=nested)
    x = randn16((m, k), seed=10 + blocks, device=device)
    (y,) = linear_forward(x, [dict(packed=packed, qs=qs)])
    assert_close(y, O.linear_ref(x.cpu().numpy(), w), what=f"{blocks} blocks, {steps} steps")


@pytest.mark.parametrize("nested", [True, False])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("blocks", [2, 4, 7, 8, 9])
def test_glu_few_steps(blocks, steps, nested, device, monkeypatch):
    """Gate and up carry code books and code2 tables of their own (halves of LDS of their own)."""
    from decik_amd.nf4 import glu_forward, launch_plan
    from decik_amd.swiglu import swiglu_fwd

    monkeypatch.setenv("DECIK_FWD_PLAN", f"{blocks},1,8")
    m, n, k = ROWS[blocks] + 1, 136, 64 * steps
    plan = launch_plan(False, m, k, [n, n], glu=True, nested=nested)
    assert plan["kernel"] == "nf4_fwd8_kernel" and plan["rows_blocks"] == blocks
    items, ws = [], []
    for i in range(2):
        p, q, w = make_weight((n, k), seed=steps + i, device=device, nested=nested)
        if i == 1:
            q.code = q.code.flip(0).contiguous()
            if nested:
                q.state2.code = q.state2.code.flip(0).contiguous()
            w = O.dequant_nf4(oracle_state(p, q), nthreads=0)
        items.append(dict(packed=p, qs=q))
        ws.append(w)
    x = randn16((m, k), seed=20 + blocks, device=device)
    g, u, h = glu_forward(x, *items)
    for out, w in zip((g, u), ws):
        assert_close(out, O.linear_ref(x.cpu().numpy(), w), what=f"{blocks} blocks, {steps} steps")
    assert torch.equal(h, swiglu_fwd(g, u))


@pytest.mark.parametrize("n", [8, 56, 64, 72, 136, 200, 320])
@pytest.mark.parametrize("blocks", [2, 4, 7, 8])
def test_input_gradient_partial_step(blocks, n, device, monkeypatch):
    """dY is a view of a wider tensor whose columns past N hold infinities and NaN."""
    from decik_amd.nf4 import linear_backward

    monkeypatch.setenv("DECIK_BWD_PLAN", f"{blocks},1")
    m, k = ROWS[blocks] + 3, 288
    packed, qs, w = make_weight((n, k), seed=n, device=device)
    wide = torch.full((m, n + 72), float("inf"), dtype=torch.float16, device=device)
    wide[:, n + 8:] = float("nan")
    dy = wide[:, :n]
    dy.copy_(randn16((m, n), seed=n + 1, device=device, std=1e-2))
    dx = linear_backward([dict(packed=packed, qs=qs, dy=dy)], m, k)
    assert_close(dx, O.linear_dx_ref(dy.contiguous().cpu().numpy(), w), what=f"{blocks} blocks, N={n}")


@pytest.mark.parametrize("plan", ["7,1", "8,1"])
@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (224, 128, 256), (257, 72, 288), (449, 200, 544)])
def test_bwd_swiglu_large_tiles(m, n, k, plan, device, monkeypatch):
    from decik_amd.nf4 import linear_backward, linear_backward_swiglu
    from decik_amd.swiglu import swiglu_bwd

    monkeypatch.setenv("DECIK_BWD_PLAN", plan)
    packed, qs, w = make_weight((n, k), seed=n + k, device=device)
    dy = randn16((m, n), seed=m, device=device, std=1e-2)
    gate, up = (randn16((m, k), seed=m + s, device=device) for s in (1, 2))
    item = dict(packed=packed, qs=qs, dy=dy)
    dg, du = linear_backward_swiglu(item, gate, up)
    grad = linear_backward([item], m, k)
    assert_close(grad, O.linear_dx_ref(dy.cpu().numpy(), w), what=f"{m}x{n}x{k}")
    dg2, du2 = swiglu_bwd(grad, gate, up)
    assert torch.equal(dg, dg2) and torch.equal(du, du2)
    g, u = gate.clone(), up.clone()  # outputs over the inputs
    dg3, du3 = linear_backward_swiglu(item, g, u, out=(g, u))
    assert torch.equal(dg3, dg) and torch.equal(du3, du)


@pytest.mark.parametrize("nested", [True, False])
@pytest.mark.parametrize("m", [9, 16, 17, 32])
@pytest.mark.parametrize("n", [8200, 16392, 20488])  # row groups of 4, 5 and 6 tiles, one round, unsplit
@pytest.mark.parametrize("k", [32, 128, 160, 1056])
def test_small_m_last_items(m, n, k, nested, device):
    from decik_amd.nf4 import launch_plan, linear_forward

    plan = launch_plan(False, m, k, [n])
    assert plan["kernel"] == "nf4_skinny_kernel" and plan["splits"] == 1
    packed, qs, w = make_weight((n, k), seed=k, device=device, nested=nested)
    x = randn16((m, k), seed=m, device=device)
    (y,) = linear_forward(x, [dict(packed=packed, qs=qs)])
    assert_close(y, O.linear_ref(x.cpu().numpy(), w), what=f"m={m} n={n} k={k}")


@pytest.mark.parametrize("m,kernel", [(9, "nf4_skinny_kernel"), (16, "nf4_skinny_kernel"),
                                      (17, "nf4_fwd"), (32, "nf4_fwd")])
@pytest.mark.parametrize("k", [32, 128, 160, 1056])
def test_small_m_two_rounds(m, kernel, k, device):
    """More than one row group a CU; past 16 rows the MFMA tiles."""
    from decik_amd.nf4 import launch_plan, linear_forward

    n = 2 ** 15 + 8
    assert launch_plan(False, m, k, [n])["kernel"].startswith(kernel)
    packed, qs, w = make_weight((n, k), seed=k, device=device)
    x = randn16((m, k), seed=m, device=device)
    (y,) = linear_forward(x, [dict(packed=packed, qs=qs)])
    assert_close(y, O.linear_ref(x.cpu().numpy(), w), what=f"m={m} k={k}")


@pytest.mark.parametrize("nested", [True, False])
@pytest.mark.parametrize("m,n,k", [
    (3, 16, 64), (16, 4872, 512), (17, 1000, 576), (32, 8968, 640),  # 1, 2, 1, 3 row tiles; 1 to 5 super-steps
    (9, 13832, 1088), (32, 18952, 1152),                            # 4, 5 row tiles; 9 super-steps
])
def test_small_m_glu_edges(m, n, k, nested, device):
    from decik_amd.nf4 import glu_forward, launch_plan
    from decik_amd.swiglu import swiglu_fwd

    assert launch_plan(False, m, k, [n, n], glu=True, nested=nested)["kernel"] == "nf4_skinny_glu_kernel"
    items, ws = [], []
    for s in range(2):
        p, q, w = make_weight((n, k), seed=n + s, device=device, nested=nested)
        items.append(dict(packed=p, qs=q))
        ws.append(w)
    x = randn16((m, k), seed=m, device=device)
    g, u, h = glu_forward(x, *items)
    for out, w in zip((g, u), ws):
        assert_close(out, O.linear_ref(x.cpu().numpy(), w), what=f"{m}x{n}x{k}")
    assert torch.equal(h, swiglu_fwd(g, u))
