"""Work splits of the flash kernels at the sizes where they can go wrong: the dispatch order of
(b, h) slices and query blocks, and the fp32 kernels' tiles, row alignment and last rows."""
import numpy as np
import pytest
import torch

from paper_01_anti_decoy_pnfirtau_amd import _lib, ops
from paper_01_anti_decoy_pnfirtau_amd.hip_pnfirtau import flash_pn_fir_tau_attention
from tests.helpers import (F32_TOL, assert_close, assert_sum_close, flash_oracle, seeded, to_np64)

pytestmark = pytest.mark.gpu


def _grads(q, k, v, tau_val, dO, causal=True):
    """O and the gradients, on leaves that keep the inputs' strides."""
    leaves = [t.detach().requires_grad_() for t in (q, k, v)]
    tau = torch.tensor(tau_val, device=q.device, requires_grad=True)
    o = flash_pn_fir_tau_attention(*leaves, tau, causal_mask=causal)
    return [o.detach(), *torch.autograd.grad(o, [*leaves, tau], dO)]


@pytest.mark.parametrize("B,H,N,D", [
    (1, 1, 300, 64), (1, 6, 300, 64), (2, 4, 257, 16), (1, 11, 300, 32), (4, 5, 130, 128),
    (67, 1, 2100, 64),   # eight whole slices per XCD in one group, and three dealt out
    (9, 3, 4100, 128),   # three per XCD in groups of two
    (33, 1, 1100, 64),   # one dealt out, ahead of the owned ones
    (6, 8, 3000, 64),    # six per XCD in one group
    (19, 8, 1100, 128),  # nineteen per XCD in three groups of seven, seven and five
])
def test_flash_slices_do_not_depend_on_the_grid(dev, B, H, N, D):
    """Every slice of a call is bitwise the slice computed alone: each (slice, block) pair is
    dispatched exactly once whatever the number of slices."""
    print(f"[flash grid B={B} H={H} N={N} D={D}]", flush=True)
    q, k, v, dO = (seeded((B, H, N, D), 500 + i, torch.bfloat16, dev) for i in range(4))
    whole = _grads(q, k, v, 0.05, dO)
    for b, h in sorted({(0, 0), (B - 1, H - 1), (B // 2, H // 2), (B // 3, 0), (0, H - 1)}):
        one = _grads(*(t[b:b + 1, h:h + 1] for t in (q, k, v)), 0.05, dO[b:b + 1, h:h + 1])
        for name, x, y in zip(("O", "dq", "dk", "dv"), whole, one):
            assert torch.equal(x[b, h], y[0, 0]), (name, b, h)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("N", [1, 15, 17, 33, 64, 65, 129, 200])
def test_flash_f32_edges_of_tiles_match_oracle(dev, N, D, aligned, causal):
    """fp32 rows that end within a 16-row block, a 32-row workgroup or a 64-row tile, from
    16-byte aligned rows and from rows that start at an odd float (staged by single floats)."""
    print(f"[flash f32 N={N} D={D} aligned={aligned} causal={causal}]", flush=True)
    B, H, tau, scale = 1, 2, 0.05, D ** -0.5
    pad = 0 if aligned else 1
    q, k, v, dO = (seeded((B, H, N, D + pad), 510 + i, torch.float32, dev)[..., pad:]
                   for i in range(4))
    o, dq, dk, dv, dt = _grads(q, k, v, tau, dO, causal)
    Of, _, _, _, rdq, rdk, rdv, rdt, dabs = flash_oracle(q, k, v, tau, dO, scale, 0.5, causal)
    for name, got, want in (("O", o, Of), ("dq", dq, rdq), ("dk", dk, rdk), ("dv", dv, rdv)):
        assert_close(to_np64(got), want, F32_TOL, F32_TOL, name)
    assert_sum_close(float(dt), rdt, dabs, F32_TOL, "dtau")


def test_flash_f32_last_value_row_not_finite(dev):
    """An infinite last row of V makes the last query's output infinite, not NaN, which the rows that
    pad the last tile by repeating it would (their weight 0 times an infinity), and reaches no query
    of another 16-key block.  (Queries that share the last row's block, 64 .. 68 here, hold its masked
    weight 0 times an infinity: NaN, as a dense product would.)"""
    N, D = 70, 64
    q, k, v, _ = (seeded((1, 1, N, D), 520 + i, torch.float32, dev) for i in range(4))
    k[..., -1, :] = q[..., -1, :]  # the last query attends to the last key
    v[..., -1, :] = float("inf")
    o = flash_pn_fir_tau_attention(q, k, v, torch.tensor(0.0, device=dev))
    assert torch.isfinite(o[..., :64, :]).all()
    assert torch.isinf(o[..., -1, :]).all()


@pytest.mark.parametrize("N", [70, 133])
def test_flash_f32_last_gradient_row_not_finite(dev, N):
    """An infinite last row of dO makes the dV of every key that the last query attends to infinite,
    not NaN: the rows that pad the last query tile by repeating it add nothing."""
    D = 64
    q, k, v, dO = (seeded((1, 1, N, D), 525 + i, torch.float32, dev).abs() for i in range(4))
    dO[..., -1, :] = float("inf")
    leaves = [t.requires_grad_() for t in (q, k, v)]
    o = flash_pn_fir_tau_attention(*leaves, torch.tensor(0.0, device=dev))
    dv = torch.autograd.grad(o, v, dO)[0]
    assert torch.isinf(dv).all()


def test_flash_f32_backward_stages_called_separately(dev):
    """The fp32 stages one by one: the dQ stage alone writes dtau, and the three together give
    bitwise the outputs of one call."""
    lib = _lib.lib()
    B, H, N, D = 1, 3, 150, 64
    q, k, v, dO = (seeded((B, H, N, D), 530 + i, torch.float32, dev) for i in range(4))
    tau = torch.tensor(0.1, device=dev)
    scale = float(1.0 / np.sqrt(D))
    o, o_lo, M, Z, _, mask = torch.ops.pnfx.flash_fwd(q, k, v, tau, scale, 0.5, True, True, False,
                                                      False)
    nws = lib.pnfx_flash_bwd_workspace_size(B, H, N, D)

    def run(stage_list):
        ws = torch.empty(nws, device=dev, dtype=torch.uint8)
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        dt = torch.zeros((), device=dev)
        for st in stage_list:
            rc = lib.pnfx_flash_bwd_stages(
                st, *ops._ptr4(q), *ops._ptr4(k), *ops._ptr4(v), *ops._ptr4(o), None,
                *ops._ptr4(dO), M.data_ptr(), Z.data_ptr(), mask.data_ptr(), *ops._ptr4(dq),
                *ops._ptr4(dk), *ops._ptr4(dv), dt.data_ptr(), ws.data_ptr(), nws, B, H, N, D,
                tau.data_ptr(), scale, 0.5, 1, 1, _lib.PNFX_F32,
                torch.cuda.current_stream().cuda_stream)
            assert rc == 0, lib.pnfx_last_error()
        torch.cuda.synchronize()
        return dq, dk, dv, dt

    one = run([_lib.PNFX_BWD_ALL])
    three = run([_lib.PNFX_BWD_PREPARE, _lib.PNFX_BWD_DQ, _lib.PNFX_BWD_DKDV])
    for name, a, b in zip(("dq", "dk", "dv"), one, three):
        assert torch.equal(a, b), name
    assert float(three[3]) == pytest.approx(float(one[3]), rel=1e-6)  # another order of fp64 sums
    dq_only = run([_lib.PNFX_BWD_PREPARE, _lib.PNFX_BWD_DQ])
    assert torch.equal(dq_only[0], one[0]) and torch.equal(dq_only[3], three[3])


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("d", [8, 20, 24, 40, 56, 72, 80, 96, 100, 104, 120])
@pytest.mark.parametrize("N,causal", [(1, True), (65, True), (300, True), (130, False)])
def test_flash_ragged_head_is_the_padded_head(dev, d, N, causal, packed):
    """Head sizes that are multiples of 8 run on the caller's rows (others padded to one), bitwise as the rows
    zero-padded to the next size with a kernel of its own: garbage in the tiles' unused columns
    (neighbouring heads' data in a packed projection) reaches nothing."""
    print(f"[flash ragged d={d} N={N} causal={causal} packed={packed}]", flush=True)
    B, H, tau, scale = 2, 3, 0.05, 0.3  # (a scale that no kernel folds into its operands)
    full = 16 if d < 16 else 32 if d < 32 else 64 if d < 64 else 128
    rows = seeded((B, N, 3, H, d), 540, torch.bfloat16, dev)
    q, k, v = (rows[:, :, i].transpose(1, 2) for i in range(3))
    if not packed:
        q, k, v = (t.contiguous() for t in (q, k, v))
    dO = seeded((B, H, N, d), 541, torch.bfloat16, dev)

    def run(*ts):
        leaves = [t.detach().requires_grad_() for t in ts[:3]]
        t0 = torch.tensor(tau, device=dev, requires_grad=True)
        o = flash_pn_fir_tau_attention(*leaves, t0, scale=scale, causal_mask=causal)
        return [o.detach(), *torch.autograd.grad(o, [*leaves, t0], ts[3])]

    got = run(q, k, v, dO)
    want = run(*(torch.nn.functional.pad(t, (0, full - d)) for t in (q, k, v, dO)))
    for name, a, b in zip(("O", "dq", "dk", "dv"), got, want):
        assert torch.equal(a, b[..., :d]), name
    assert torch.equal(got[4], want[4])


@pytest.mark.parametrize("d", [8, 24, 40, 56, 80, 104])
def test_flash_ragged_head_skips_silent_keys(dev, d):
    """Blocks of zero keys under tau > 0, at a size where the forward takes the silent-tile bound (key
    norms over the d columns that exist, heads up to 64): bitwise the zero-padded rows, tile mask
    included, and the bound does skip (no positive score in those blocks)."""
    print(f"[flash ragged silent d={d}]", flush=True)
    B, H, N = 4, 4, 2080
    full = 16 if d < 16 else 32 if d < 32 else 64 if d < 64 else 128
    q, k, v, dO = (seeded((B, H, N, d), 560 + i, torch.bfloat16, dev) for i in range(4))
    for j in range(0, N, 128):
        k[:, :, j:j + 64] = 0
    tau, scale = torch.tensor(0.25, device=dev), 0.3
    assert B * H * N * N >= 1 << 26  # the op takes the bound from here on

    def run(*ts):
        o, o_lo, M, Z, _, mask = torch.ops.pnfx.flash_fwd(*ts[:3], tau, scale, 0.5, True, True, False,
                                                          False)
        grads = torch.ops.pnfx.flash_bwd(*ts[:3], tau, o, o_lo, ts[3], M, Z, mask, scale, 0.5, True,
                                         True)
        return [o, *grads[:3]], [M, Z, mask, grads[3]]

    (got, gs), (want, ws) = run(q, k, v, dO), run(*(torch.nn.functional.pad(t, (0, full - d))
                                                    for t in (q, k, v, dO)))
    for a, b in zip(got, want):
        assert torch.equal(a, b[..., :d])
    for a, b in zip(gs, ws):
        assert torch.equal(a, b)
    assert not gs[2][:, :, 0::2].any() and gs[2][:, -1, 1:-1:2].all()


@pytest.mark.parametrize("d", [8, 24, 40, 72, 80, 120])
def test_flash_ragged_head_infinite_key_stays_visible(dev, d):
    """An infinite key entry in the last columns of a ragged head: O and dq are finite exactly where
    those of the zero-padded rows with one kernel size more are (a query that scores +inf against the
    key is not, and the key is not dropped)."""
    print(f"[flash ragged inf d={d}]", flush=True)
    B, H, N = 1, 2, 150
    full = 32 if d < 32 else 64 if d < 64 else 128
    q, k, v, dO = (seeded((B, H, N, d), 550 + i, torch.bfloat16, dev) for i in range(4))
    k[0, 0, 37, d - 1] = float("inf")

    def run(*ts):
        t0 = torch.tensor(0.0, device=dev)
        leaves = [t.detach().requires_grad_() for t in ts[:3]]
        o = flash_pn_fir_tau_attention(*leaves, t0, scale=0.3)
        return o.detach(), torch.autograd.grad(o, leaves[0], ts[3])[0]

    got = run(q, k, v, dO)
    want = run(*(torch.nn.functional.pad(t, (0, full - d)) for t in (q, k, v, dO)))
    for a, b in zip(got, want):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b[..., :d]))
    hit = (q[0, 0, :, d - 1] > 0) & (torch.arange(N, device=dev) >= 37)
    assert torch.equal(torch.isfinite(got[0]).all(-1)[0, 0], ~hit) and hit.any()
    assert torch.isfinite(got[0][0, 1]).all()
