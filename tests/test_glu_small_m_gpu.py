"""The fused gate+up+SwiGLU forward at 1-32 token rows (the GEMV's and the small-M kernel's GLU
forms, MFMA tiles beyond): gate and up against the oracle, h the SwiGLU kernel's bits on them, the
outputs optional, at the sizes where the forms' tiles end and where the dispatch changes. Gate and
up carry code books and code2 tables of their own."""

import pytest
import torch

from helpers import assert_close, make_weight, oracle_state, randn16
from oracle import nf4 as O

pytestmark = pytest.mark.gpu

CASES = [
    # (m, n, k, blocksize, nested, kernel); row tiles: of each weight, a work-group
    (1, 8, 64, 64, True, "nf4_gemv_kernel"),               # one work-group, one chunk pair a row
    (1, 1544, 3584, 64, True, "nf4_gemv_kernel"),          # several loads a thread, a ragged last group
    (1, 40, 20480, 128, False, "nf4_gemv_kernel"),         # long rows: several loads a row
    (2, 264, 1536, 64, True, "nf4_skinny_glu_kernel"),     # two rows of short contractions
    (2, 264, 2048, 64, True, "nf4_gemv_kernel"),           # ... and of longer ones
    (2, 2056, 2048, 64, True, "nf4_skinny_glu_kernel"),    # more rows than the GEMV takes
    (2, 72, 8960, 64, False, "nf4_gemv_kernel"),
    (3, 8, 64, 64, True, "nf4_skinny_glu_kernel"),         # fewer rows than a tile, half a super-step
    (3, 4864, 896, 64, True, "nf4_skinny_glu_kernel"),     # 2 row tiles
    (16, 8968, 192, 64, True, "nf4_skinny_glu_kernel"),    # 3 row tiles, a ragged last group
    (8, 12296, 128, 64, False, "nf4_skinny_glu_kernel"),   # 4 row tiles: 8 rows more than 3 would take
    (5, 18952, 256, 128, True, "nf4_skinny_glu_kernel"),   # 5 row tiles
    (17, 1032, 1536, 64, True, "nf4_skinny_glu_kernel"),   # two token blocks
    (32, 12296, 128, 64, False, "nf4_skinny_glu_kernel"),  # two token blocks, 4 row tiles
    (11, 28680, 128, 64, True, "nf4_skinny_glu_kernel"),   # two rounds of work-groups
    (12, 28680, 128, 64, True, "nf4_fwd8_kernel"),         # ... which from here on outlast the MFMA tiles
]


@pytest.mark.parametrize("m,n,k,blocksize,nested,kernel", CASES)
def test_glu_few_rows(m, n, k, blocksize, nested, kernel, device):
    from decik_amd.nf4 import glu_forward, launch_plan, linear_forward
    from decik_amd.swiglu import swiglu_fwd

    assert launch_plan(False, m, k, [n, n], glu=True, nested=nested, blocksize=blocksize)["kernel"] == kernel
    weights = []
    for i in range(2):
        p, q, w = make_weight((n, k), seed=n + k + i, device=device, blocksize=blocksize, nested=nested)
        if i == 1:
            q.code = q.code.flip(0).contiguous()
            if nested:
                q.state2.code = q.state2.code.flip(0).contiguous()
            w = O.dequant_nf4(oracle_state(p, q), nthreads=0)
        weights.append((dict(packed=p, qs=q, bias=randn16((n,), seed=7 + i, device=device, std=0.1)), w))
    x = randn16((m, k), seed=m, device=device)
    g, u, h = glu_forward(x, weights[0][0], weights[1][0])
    for out, (it, w) in zip((g, u), weights):
        # fp32 sums, one fp16 rounding: the GEMM bar
        assert_close(out, O.linear_ref(x.cpu().numpy(), w, it["bias"].cpu().numpy()), what=f"{m}x{n}x{k}")
    assert torch.equal(h, swiglu_fwd(g, u))
    assert torch.equal(glu_forward(x, weights[0][0], weights[1][0], keep_gate_up=False)[2], h)
    if m == 1:  # the GEMV's sums depend on k only: the grouped launch's bits
        g2, u2 = linear_forward(x, [weights[0][0], weights[1][0]])
        assert torch.equal(g, g2) and torch.equal(u, u2)


@pytest.mark.parametrize("m", [1, 2, 3, 16, 17, 32])
def test_glu_few_rows_precision(m, device, monkeypatch):
    """The few-row forms' sums are no worse than the MFMA tiles': the gate and up values that are not
    the correctly rounded 64-bit sums, counted for both on the same inputs. Bound: the tiles' count
    and three standard deviations of such a (Poisson) count."""
    from decik_amd.nf4 import glu_forward

    n, k = 8960, 1536
    items, exact = [], []
    x = randn16((m, k), seed=m, device=device)
    for i in range(2):
        p, q, w = make_weight((n, k), seed=40 + i, device=device)
        items.append(dict(packed=p, qs=q))
        exact.append((x.double().cpu() @ torch.from_numpy(w).double().T).half())
    def misrounded():
        return sum(int((y.cpu() != e).sum()) for y, e in zip(glu_forward(x, *items)[:2], exact))
    few = misrounded()
    monkeypatch.setenv("DECIK_FWD_PLAN", "2,1,8")
    tiles = misrounded()
    assert tiles > 0 and few <= tiles + 3 * tiles ** 0.5, (few, tiles)


@pytest.mark.parametrize("m,n", [(1, 64), (4, 200), (20, 200)])
def test_glu_few_rows_strided(m, n, device):
    """X and every output as rows of wider buffers; what lies beside them is not touched."""
    from decik_amd._lib import LinearFwdGroup, check, lib, ptr, stream_of, weight_desc
    from decik_amd.nf4 import glu_forward

    k, pad = 320, 24
    items = [make_weight((n, k), seed=i, device=device)[:2] for i in range(2)]
    xw = randn16((m, k + pad), seed=5, device=device)
    want = glu_forward(xw[:, :k].contiguous(), *(dict(packed=p, qs=q) for p, q in items))
    outs = [torch.full((m, n + pad), 7.0, dtype=torch.float16, device=device) for _ in range(3)]
    groups, keep = (LinearFwdGroup * 2)(), []
    for i, (p, q) in enumerate(items):
        groups[i].w, kp = weight_desc(p, q, device)
        groups[i].y, groups[i].ldy = outs[i].data_ptr(), n + pad
        keep.append(kp)
    check(lib().dk_nf4_glu_fwd(ptr(xw), m, k, k + pad, groups, 0, ptr(outs[2]), n + pad, stream_of(device)))
    for out, ref in zip(outs, want):
        assert torch.equal(out[:, :n], ref) and bool((out[:, n:] == 7.0).all())


@pytest.mark.parametrize("m,n,k", [(1, 264, 576), (2, 264, 2112), (3, 264, 576), (20, 264, 576)])
@pytest.mark.parametrize("nested", [True, False])
def test_glu_few_rows_optional_operands(m, n, k, nested, device):
    """One output and one bias at a time, and token rows of infinities and NaN, which stay in their
    rows (rows past m, the contraction's tail and weight rows past n read as zeros beside them)."""
    from decik_amd._lib import LinearFwdGroup, check, lib, ptr, stream_of, weight_desc
    from decik_amd.nf4 import glu_forward

    items = [make_weight((n, k), seed=30 + i, device=device, nested=nested)[:2] for i in range(2)]
    bias = randn16((n,), seed=9, device=device, std=0.2)
    x = randn16((m, k), seed=m, device=device)
    for which in range(2):
        dicts = [dict(packed=p, qs=q, bias=bias if i == which else None) for i, (p, q) in enumerate(items)]
        want = glu_forward(x, *dicts)
        y, h = (torch.full((m, n), 7.0, dtype=torch.float16, device=device) for _ in range(2))
        groups, keep = (LinearFwdGroup * 2)(), []
        for i, (p, q) in enumerate(items):
            groups[i].w, kp = weight_desc(p, q, device)
            keep.append(kp)
        groups[which].y, groups[which].ldy, groups[which].bias = y.data_ptr(), n, bias.data_ptr()
        check(lib().dk_nf4_glu_fwd(ptr(x), m, k, k, groups, 0, ptr(h), n, stream_of(device)))
        assert torch.equal(y, want[which]) and torch.equal(h, want[2])
    for bad in (float("inf"), float("nan")):
        xb = x.clone()
        xb[m - 1] = bad
        out = glu_forward(xb, *dicts)
        for a, b in zip(out, want):
            assert torch.equal(a[:m - 1], b[:m - 1]) and not bool(torch.isfinite(a[m - 1]).any())
