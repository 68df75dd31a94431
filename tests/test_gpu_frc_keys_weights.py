"""frc_from_keys at the edges of its lane groups and row blocks, and with
weights S_j = r_j / (r_j + 1e-8) that are 1 in fp32 (the second Gram pass then
leaves at once) and that are not (a key whose norm the floor of 1e-12 cuts)."""

import numpy as np
import pytest
import torch

from oracle import cab_oracle as O

pytestmark = pytest.mark.gpu


def _check(cuda, keys):
    from cab_attention.kernels import frc_from_keys
    got = {k: x.double().cpu().numpy() for k, x in frc_from_keys(keys.to(cuda), return_parts=True).items()}
    want = O.frc_from_keys(keys.double().numpy())
    # Each product of split operands is within 2e-5 of its terms' magnitudes
    # (2^-16, dropped lo x lo included), fp32 sums within 1e-6.
    x = keys.double().numpy().mean(axis=(0, 1))
    kn = x / np.maximum(np.linalg.norm(x, axis=-1, keepdims=True), 1e-12)
    bound = 2e-5 * np.abs(kn @ kn.T).sum(axis=1) + 1e-6
    r = want["row_sums"]
    assert np.all(np.abs(got["row_sums"] - r) <= bound)
    ok = r > 1e-3  # a cut key's ratios hang on its own rounding
    np.testing.assert_allclose(got["strengths"][ok], want["strengths"][ok], atol=1e-5, rtol=0)
    tol = 2 * bound / np.maximum(r, 1e-30) + 2e-6
    assert np.all(np.abs(got["triangles"] - want["triangles"])[ok] <= tol[ok])
    assert np.all(np.abs(got["frc"] - want["frc"])[ok] <= 3 * tol[ok] + 2e-5)
    zero = r == 0
    for name in ("strengths", "triangles", "frc", "row_sums"):
        assert np.all(got[name][zero] == 0)


@pytest.mark.parametrize("B,H,N,D", [(1, 1, 255, 8), (1, 3, 256, 64), (1, 5, 257, 72), (3, 3, 513, 128),
                                     (1, 9, 300, 136), (2, 2, 40, 256)])
@pytest.mark.parametrize("cut", [False, True])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_frc_from_keys_weights(cuda, B, H, N, D, cut, dt):
    g = torch.Generator().manual_seed(N + D)
    keys = torch.randn((B, H, N, D), generator=g) + 0.3
    if cut:
        keys[:, :, N // 2] *= 1e-14  # kn = x / 1e-12: r_j about 1e-2, S_j below 1
        keys[:, :, 3] = 0.0
    _check(cuda, keys.to(dt))
