"""The guide's staged layer inputs and deltas (blocks of 16 samples) at the
sizes where a block, a 32-sample step or a slice of the weight-gradient sum is
partly filled or empty.  Both operands of a weight gradient are BF16 (rounding
2^-9 each), so 1e-2 relative (Frobenius) leaves a factor of two."""
import numpy as np
import pytest
import torch

import oracle_bind as ob
from guide_util import b_off, random_params, random_samples, w_off

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 33, 1000, 1056])
def test_gradient_at_block_edges(gpu_ctx, n):
    import wayland_amd as wl
    print(f"case: guide staging n={n}", flush=True)
    P = random_params(51)
    g = wl.Guide(gpu_ctx, batch_size=1056)
    g.set_params(P.astype(np.float32))
    dev = lambda a: torch.as_tensor(a, dtype=torch.float32, device="cuda").contiguous()  # noqa: E731
    g.gradient(dev(random_samples(53, 1056)))  # rows that a smaller batch must not see
    S = random_samples(52, n)
    grad = g.gradient(dev(S))[0].cpu().numpy()
    ref = ob.guide_loss_grad(P.astype(np.float32).astype(np.float64), S, emulate_bf16=True)[1]
    for l in range(5):
        n_out = 64 if l < 4 else 32
        for sl in (slice(w_off(l), b_off(l)), slice(b_off(l), b_off(l) + n_out)):
            e = np.linalg.norm(grad[sl] - ref[sl]) / np.linalg.norm(ref[sl])
            assert e < 1e-2
    g.close()
