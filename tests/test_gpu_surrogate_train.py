"""The training kernel's rounds and remainders: fewer samples than a wave, a workgroup and its round, a
partial last workgroup, and more rounds than one per workgroup (16,385 samples over 256 workgroups of 64),
with and without weights, against the FP64 oracle with the same operand rounding: per parameter block
relative L2 < 1e-2, as the training kernel's other test (operands that land next to a rounding boundary
round the other way than FP64's, one 16-bit unit, 1e-3 (FP16) to 8e-3 (BF16), of a few of the sums' terms)."""
import numpy as np
import pytest

from oracle import mlp
from skyrendering_amd import surrogate as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("network", ["f16_gate", "bf16_silu"])
@pytest.mark.parametrize("n,weighted", [(1, True), (15, False), (64, True), (65, True), (1000, False), (16385, True)])
def test_gradient_sizes_match_oracle(ctx, network, n, weighted):
    rng = np.random.default_rng(n)
    p = sg.init_params(3).astype(np.float32)
    f = np.zeros((n, 8), np.float32)
    f[:, :7] = rng.uniform(-1, 1, size=(n, 7))
    t = rng.normal(-2.0, 1.0, size=(n, 3)).astype(np.float32)
    w = rng.uniform(0.1, 1.0, n).astype(np.float32) if weighted else None
    model = sg.SkySurrogate(ctx, p, network=network)
    fd, td = ctx.upload(f), ctx.upload(t)
    wd = ctx.upload(w) if weighted else None
    scale = 1.0 / (3 * n)
    for _ in range(2):  # the second call reuses the workspace
        model.gradient(fd.ptr, td.ptr, n, scale, wd.ptr if weighted else None)
    g = model.grad.download(np.float32, (sg.PARAMS,)).astype(np.float64)
    loss = float(model.loss.download(np.float32, (1,))[0])
    ref_loss, ref = mlp.loss_and_grad(p.astype(np.float64), f.astype(np.float64), t.astype(np.float64), scale,
                                      network=network, rounded=True, weights=w)
    assert abs(loss - ref_loss) < 1e-3 * ref_loss
    at = 0
    for k, m in sg.LAYERS:
        for size in (m * k, m):
            a, b = g[at:at + size], ref[at:at + size]
            assert np.linalg.norm(a - b) < 1e-2 * np.linalg.norm(b), (k, m, size)
            at += size
