"""The training and inference kernels' tiles at their edges: rows around a 16-row tile, a
workgroup's four tiles and the 256 workgroups of a batch, against the FP64 oracle."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from realtimeparticles_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 16383, 16385, 40001])
def test_tiles_match_fp64_oracle_and_repeat(n):
    rng = np.random.default_rng(n)
    p = rng.normal(0, 0.3, MO.N_PARAMS).astype(np.float32)
    feat = rng.normal(0, 1.5, (n, 8)).astype(np.float32)
    target = rng.normal(0, 2.0, n).astype(np.float32)
    mu = rng.normal(0, 0.2, 8).astype(np.float32)
    sigma = rng.uniform(0.5, 2.0, 8).astype(np.float32)
    m = capi.Mlp()
    m.set_params(p)
    m.set_normalization(mu, sigma, 2.0)
    grad, loss = m.gradients(feat, target)
    again, loss2 = m.gradients(feat, target)
    assert np.array_equal(grad, again) and loss == loss2
    ref, ref_loss = MO.gradients(p, feat, target, mu, sigma, 2.0, bf16_ops=True)
    # FP32 against FP64 sums move some operands to the other bf16 neighbour, 2^-8 of the
    # operand at most, and every product is linear in its operands
    assert loss == pytest.approx(ref_loss, rel=2.0 ** -7)
    for a, b in ((0, 512), (512, 576), (576, 4672), (4672, 4736), (4736, 4800), (4800, 4801)):
        assert np.linalg.norm(grad[a:b] - ref[a:b]) <= 2.0 ** -7 * np.linalg.norm(ref[a:b])
    out = m.forward(feat).astype(np.float64)
    ref_out, _ = MO.forward(p, feat, mu, sigma, 2.0, bf16_ops=True)
    assert np.all(np.abs(out - ref_out) <= 1e-2 * (1.0 + np.abs(ref_out)))
    m.close()
