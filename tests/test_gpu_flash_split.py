"""Work splits of the flash kernels at the sizes where they can go wrong: the dispatch order of
(b, h) slices and query blocks."""
import pytest
import torch

from paper_01_anti_decoy_pnfirtau_amd.hip_pnfirtau import flash_pn_fir_tau_attention
from tests.helpers import seeded

pytestmark = pytest.mark.gpu


def _grads(q, k, v, tau_val, dO, causal=True):
    """O and the gradients, on leaves that keep the inputs' strides."""
    leaves = [t.detach().requires_grad_() for t in (q, k, v)]
    tau = torch.tensor(tau_val, device=q.device, requires_grad=True)
    o = flash_pn_fir_tau_attention(*leaves, tau, causal_mask=causal)
    return [o.detach(), *torch.autograd.grad(o, [*leaves, tau], dO)]


@pytest.mark.parametrize("B,H,N,D", [
    (1, 1, 300, 64), (1, 6, 300, 64), (2, 4, 257, 16), (1, 11, 300, 32), (4, 5, 130, 128),
    (67, 1, 2100, 64),   # eight whole slices per XCD in groups of seven, and three dealt out
    (9, 3, 4100, 128),   # three per XCD in groups of two
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
