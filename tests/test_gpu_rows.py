"""GPU parity of the row-fused score kernels against the oracle (src/triton_pnfirtau.py:141-303)."""
import numpy as np
import pytest
import torch

from oracle import pnfirtau_oracle as O
from paper_01_anti_decoy_pnfirtau_amd import ops  # noqa: F401  (registers torch.ops.pnfx)
from tests.helpers import BF16_ATOL, F32_TOL, assert_bf16_close, assert_close, seeded, to_np64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,causal,p,gamma", [(24, True, 10.0, 0.5), (130, True, 10.0, 0.5),
                                              (64, False, 2.0, None), (50, True, 3.5, 0.75),
                                              (512, True, 10.0, 0.5), (5000, True, 10.0, 0.5)])
def test_rows_fwd_bwd_match_oracle(dev, dtype, N, causal, p, gamma):
    print(f"[rows N={N} causal={causal} p={p} gamma={gamma} {dtype}]", flush=True)
    B, H = (2, 2) if N < 1000 else (1, 1)
    raw = seeded((B, H, N, N), 10, dtype, dev, scale=3.0)
    if N >= 24:
        raw[0, 0, 20, :5] = raw[0, 0, 20, 7]  # planted tie at the row peak candidates
    tau = torch.tensor(0.3, device=dev, requires_grad=True)
    scale = 0.25
    rawg = raw.clone().requires_grad_(True)
    from paper_01_anti_decoy_pnfirtau_amd.hip_pnfirtau import hip_pn_fir_tau_scores
    w = hip_pn_fir_tau_scores(rawg, tau, scale=scale, p=p, gamma=gamma, causal_mask=causal)
    dW = seeded(w.shape, 11, dtype, dev)
    w.backward(dW)
    torch.cuda.synchronize()
    rn = to_np64(raw)
    W, M, Z, Nm = O.pn_rows_fwd(rn, 0.3, scale, p, gamma, causal)
    d_raw, dtr = O.pn_rows_bwd(to_np64(dW), rn, 0.3, M, Z, Nm, scale, p, gamma, causal)
    if dtype == torch.float32:  # fp32 bar: 1e-5 (rtol, and atol of the tensor's scale)
        assert_close(to_np64(w), W, F32_TOL, F32_TOL, "W")
        assert_close(to_np64(rawg.grad), d_raw, F32_TOL, F32_TOL, "d_raw")
        tol = F32_TOL
    else:
        assert_bf16_close(to_np64(w), W, "W")
        assert_bf16_close(to_np64(rawg.grad), d_raw, "d_raw")
        tol = BF16_ATOL
    assert abs(float(tau.grad) - dtr.sum()) <= tol * max(1.0, np.abs(dtr).sum())


def test_rows_stats_and_silent_rows(dev):
    raw = seeded((1, 1, 40, 40), 12, torch.float32, dev)
    raw[0, 0, 10] = -5.0  # silent row
    raw[0, 0, 30, :4] = 3.0  # four-way tie at the peak
    tau = torch.tensor(0.1, device=dev)
    w, M, Z, Nm = torch.ops.pnfx.pn_rows_fwd(raw, tau, 1.0, 10.0, 0.5, True, True)
    Wo, Mo, Zo, No = O.pn_rows_fwd(to_np64(raw), 0.1, 1.0, 10.0, 0.5, True)
    assert np.array_equal(Nm.cpu().numpy(), No.reshape(-1))
    assert float(M[10]) == 0.0 and float(Z[10]) == pytest.approx(1e-12) and int(Nm[10]) == 0
    assert int(Nm[30]) == 4
    assert torch.all(w[0, 0, 10] == 0)
    np.testing.assert_allclose(M.cpu().numpy(), Mo.reshape(-1), rtol=1e-6)
    np.testing.assert_allclose(Z.cpu().numpy(), Zo.reshape(-1), rtol=1e-5)
    # row sums equal gate * mass / (mass + 1e-12), i.e. the gate unless the mass is tiny
    np.testing.assert_allclose(w.sum(-1).cpu().numpy().reshape(-1), Wo.sum(-1).reshape(-1), rtol=1e-5, atol=1e-7)


def test_rows_of_length_one_and_many_rows(dev):
    """Score rows of one key (the row's only score is its peak) and a tall stack of short rows."""
    for shape in ((3, 5, 1, 1), (20000, 3, 3)):
        raw = torch.randn(shape, device=dev).to(torch.bfloat16)
        print(f"[rows {tuple(raw.shape)}]", flush=True)
        tau = torch.tensor(0.1, device=dev)
        w, M, Z, Nm = torch.ops.pnfx.pn_rows_fwd(raw, tau, 0.5, 10.0, 0.5, True, False)
        s = raw.float() * 0.5 - 0.1
        u = s.clamp_min(0)
        P = (u ** 10)
        m = u.amax(-1, keepdim=True)
        g = torch.where(m > 0, m / (m + 0.5), torch.zeros_like(m))
        ref = P / (P.sum(-1, keepdim=True) + 1e-12) * g
        torch.testing.assert_close(w.float(), ref, rtol=2e-2, atol=2e-3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("p", [10.0, 2.0, 3.5])
@pytest.mark.parametrize("N", [1, 7, 9, 63, 65, 127, 129, 255, 257, 383, 385, 511, 513, 1023, 1025, 2051])
def test_rows_ends_of_chunks_match_oracle(dev, dtype, N, p):
    """Rows that start at any element and end within a 16-byte chunk, one to five register chunks
    long, forward and backward; short bf16 rows that go by elements, one to six registers long."""
    print(f"[rows N={N} p={p} {dtype}]", flush=True)
    from paper_01_anti_decoy_pnfirtau_amd.hip_pnfirtau import hip_pn_fir_tau_scores
    raw = seeded((1, 1, N, N), 30, dtype, dev, scale=2.0).requires_grad_()
    dW = seeded((1, 1, N, N), 31, dtype, dev)
    tau = torch.tensor(0.1, device=dev, requires_grad=True)
    w = hip_pn_fir_tau_scores(raw, tau, scale=0.5, p=p, gamma=0.5, causal_mask=True)
    w.backward(dW)
    rn = to_np64(raw)
    W, M, Z, Nm = O.pn_rows_fwd(rn, 0.1, 0.5, p, 0.5, True)
    d_raw, dtr = O.pn_rows_bwd(to_np64(dW), rn, 0.1, M, Z, Nm, 0.5, p, 0.5, True)
    if dtype == torch.float32:
        assert_close(to_np64(w), W, F32_TOL, F32_TOL, "W")
        assert_close(to_np64(raw.grad), d_raw, F32_TOL, F32_TOL, "d_raw")
    else:
        assert_bf16_close(to_np64(w), W, "W")
        assert_bf16_close(to_np64(raw.grad), d_raw, "d_raw")
    tol = F32_TOL if dtype == torch.float32 else BF16_ATOL
    assert abs(float(tau.grad) - dtr.sum()) <= tol * max(1.0, np.abs(dtr).sum())


@pytest.mark.parametrize("p,size", [(10.0, 1e-6), (10.0, 1e-4), (10.0, 1e-3), (10.0, 1e3), (2.0, 1e-12),
                                    (2.0, 1e12)])
def test_rows_backward_over_the_range_of_peaks(dev, p, size):
    """The backward's power-of-two unit: peaks whose powers are far from 1, or below fp32's range
    (the largest scores here are 4.4 times `size`: at 1e3 their tenth powers end at 3e36, and 7e3
    overflows fp32 in the forward; at 1e-6 the gradients end below 1e-40)."""
    from paper_01_anti_decoy_pnfirtau_amd.hip_pnfirtau import hip_pn_fir_tau_scores
    N = 96
    raw = (seeded((1, 1, N, N), 32, torch.float32, dev).abs() * size).requires_grad_()
    dW = seeded((1, 1, N, N), 33, torch.float32, dev)
    tau = torch.tensor(0.0, device=dev, requires_grad=True)
    w = hip_pn_fir_tau_scores(raw, tau, scale=1.0, p=p, gamma=0.5, causal_mask=True)
    w.backward(dW)
    rn = to_np64(raw)
    W, M, Z, Nm = O.pn_rows_fwd(rn, 0.0, 1.0, p, 0.5, True)
    d_raw, dtr = O.pn_rows_bwd(to_np64(dW), rn, 0.0, M, Z, Nm, 1.0, p, 0.5, True)
    if np.abs(d_raw).max() < 2.0 ** -126:  # nothing that fp32 holds as a normal number
        for t in (w, raw.grad, tau.grad):
            assert float(t.detach().abs().max()) < 2.0 ** -126
        return
    assert np.abs(d_raw).max() > 1e-28 and np.abs(W).max() > 1e-28  # assert_close's floor is 1e-30
    assert_close(to_np64(w), W, F32_TOL, F32_TOL, "W")
    # nine roundings of u^9 and those of dW - D: 2e-5 of the largest entry
    assert_close(to_np64(raw.grad), d_raw, 2 * F32_TOL, 2 * F32_TOL, "d_raw")
    # a sum of row sums: the entries' own errors of 2e-5 of their size
    assert abs(float(tau.grad) - dtr.sum()) <= 2 * F32_TOL * np.abs(d_raw).sum()


@pytest.mark.parametrize("n", [1, 3, 5, 4096, 16385, 131072, 131073, 400001])
def test_sum_f64_is_the_double_sum(dev, n):
    """pnfx::sum_f64 (the tau gradient from the row partials): one and two launches, odd lengths,
    and a view that does not start on 16 bytes; fp64 sums agree to their own rounding."""
    x = seeded((n + 1,), 34, torch.float32, dev)
    for t in (x[:n], x[1:]):
        want = float(t.double().sum())
        bound = 1e-14 * float(t.double().abs().sum())
        assert abs(float(torch.ops.pnfx.sum_f64(t, True)) - want) <= bound
        got = torch.ops.pnfx.sum_f64(t, False)
        assert got.dtype == torch.float32 and abs(float(got) - want) <= 6e-8 * abs(want) + bound


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N", [31, 64, 777, 2100])
def test_rows_masked_weight_gradients_reach_nothing(dev, dtype, N):
    """Infinities and NaN of dW past the causal limit, in the 16-byte chunk that straddles it and after
    it: the gradients of the same call with zeros there, bit for bit."""
    raw = seeded((1, 1, N, N), 35, dtype, dev, scale=2.0)
    dW = seeded((1, 1, N, N), 36, dtype, dev).tril_()
    bad = torch.full_like(dW, float("inf"))
    bad[..., 1::2] = float("nan")
    tau = torch.tensor(0.1, device=dev)
    for p in (10.0, 2.0, 3.5):
        w, M, Z, Nm = torch.ops.pnfx.pn_rows_fwd(raw, tau, 0.5, p, 0.5, True, True)
        want = torch.ops.pnfx.pn_rows_bwd(dW, raw, tau, M, Z, Nm, 0.5, p, 0.5, True, True)
        got = torch.ops.pnfx.pn_rows_bwd(dW + bad.triu(1), raw, tau, M, Z, Nm, 0.5, p, 0.5, True, True)
        assert all(torch.equal(a, b) and torch.isfinite(a).all() for a, b in zip(got, want)), p


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("p,big", [(10.0, 1e4), (2.0, 1e20), (3.5, 1e12)])
@pytest.mark.parametrize("N", [64, 95])
def test_rows_overflow_of_the_powers_stays_visible(dev, dtype, p, big, N):
    """A row whose largest score's power overflows fp32 has NaN in W, and NaN for the gradient of each
    of its positive scores and of tau, not zeros; the other rows are those of the call without it."""
    raw = seeded((1, 1, N, N), 37, dtype, dev)
    dW = seeded((1, 1, N, N), 38, dtype, dev)
    tau = torch.tensor(0.0, device=dev)
    res = []
    for spike in (None, big):
        r = raw.clone()
        if spike:
            r[0, 0, 40, 7] = spike
        w, M, Z, Nm = torch.ops.pnfx.pn_rows_fwd(r, tau, 1.0, p, 0.5, True, True)
        d, dt = torch.ops.pnfx.pn_rows_bwd(dW, r, tau, M, Z, Nm, 1.0, p, 0.5, True, True)
        res.append((w[0, 0], d[0, 0], dt, r[0, 0]))
    (w0, d0, t0, _), (w, d, t, r) = res
    others = torch.arange(N, device=dev) != 40
    assert all(torch.equal(a[others], b[others]) for a, b in ((w, w0), (d, d0), (t, t0)))
    on = (r[40] > 0) & (torch.arange(N, device=dev) <= 40)
    assert torch.isnan(w[40, 7]) and torch.isnan(t[40])
    assert torch.equal(torch.isnan(d[40]), on) and bool((d[40][~on] == 0).all())
