"""compute_block_frc at M <= 128 (one kernel) and above (the general ones: the
affinity's runs of four columns whole and cut), at the edges of 32-wide tiles and 16-deep k-steps, every input type and
formula it takes, with and without diagnostics, against the oracle."""

import numpy as np
import pytest
import torch

from oracle import cab_oracle as O

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


@pytest.mark.parametrize("M,D", [(1, 128), (2, 8), (31, 64), (32, 24), (33, 128), (64, 256), (65, 72),
                                 (100, 128), (127, 64), (128, 128), (129, 128),
                                 (130, 64), (131, 128), (132, 72), (255, 128)])
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("formula", ["additive", "multiplicative"])
def test_frc_small(cuda, M, D, dt, formula):
    from cab_attention.kernels import compute_block_frc
    g = torch.Generator().manual_seed(M * 131 + D)
    qc, kc = (torch.randn((2, 3, M, D), generator=g).to(DTYPES[dt]) for _ in range(2))
    frc, aff, tri = compute_block_frc(qc.to(cuda), kc.to(cuda), lambda_redundancy=0.7, formula=formula)
    only, none_a, none_t = compute_block_frc(qc.to(cuda), kc.to(cuda), lambda_redundancy=0.7,
                                             formula=formula, diagnostics=False)
    assert none_a is None and none_t is None
    f, a, t = (x.double().cpu().numpy() for x in (frc, aff, tri))
    wf, wa, wt = O.compute_block_frc(qc.float().numpy(), kc.float().numpy(), lambda_redundancy=0.7,
                                     formula=formula)
    np.testing.assert_allclose(a, wa, rtol=1e-4, atol=2e-6)
    assert np.all((a == 0) == (np.asarray(wa) == 0))  # the minimum maps to exactly 0
    # T: f16 products, 2 x 2^-11 a term; F: that error times lambda (additive)
    bound = 1e-3 * np.asarray(wt) + 1e-6
    assert np.all(np.abs(t - wt) <= bound)
    for got in (f, only.double().cpu().numpy()):
        if formula == "additive":
            assert np.all(np.abs(got - wf) <= 0.7 * bound + 1e-3 * np.abs(wa) + 1e-6)
        else:
            # d/dT of Ahat / (1 + lambda T / (Ahat + 1e-8)) is at most F / T
            assert np.all(np.abs(got - wf) <= 2e-3 * np.abs(wf) + 1e-6)


def test_constant_affinity(cuda):
    """min == max: A is left as it is, far outside fp16's range here, and T = M c^2."""
    from cab_attention.kernels import compute_block_frc
    q = torch.full((1, 1, 50, 64), 300.0)
    frc, aff, tri = compute_block_frc(q.to(cuda), q.to(cuda))
    c = 300.0 * 300.0 * 64 / 8.0
    torch.testing.assert_close(aff.cpu(), torch.full((1, 1, 50, 50), c))
    torch.testing.assert_close(tri.cpu(), torch.full((1, 1, 50, 50), 50 * c * c))
    torch.testing.assert_close(frc.cpu(), torch.full((1, 1, 50, 50), c - 0.5 * 50 * c * c))


@pytest.mark.parametrize("M", [16, 33, 100, 128, 129])
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
def test_fused_form_has_one_set_of_roundings(cuda, M, dt):
    """Without diagnostics F = X (I - lambda X)^T of fp16 planes, at M <= 128 as
    above it: blocks at the selection's threshold do not depend on M's side of 128."""
    from cab_attention.kernels import compute_block_frc
    g = torch.Generator().manual_seed(M)
    qc, kc = (torch.randn((1, 2, M, 64), generator=g).to(DTYPES[dt]).to(cuda) for _ in range(2))
    lam = float(np.float32(0.7))
    _, aff, _ = compute_block_frc(qc, kc, lambda_redundancy=lam)
    frc, _, _ = compute_block_frc(qc, kc, lambda_redundancy=lam, diagnostics=False)
    a = aff.cpu().double()
    x = a.half().double()
    xt = (torch.eye(M, dtype=torch.float64) - lam * a).half().double()  # [k][j], rounded once
    want = torch.matmul(x, xt)
    bound = M * 2.0 ** -23 * torch.matmul(x.abs(), xt.abs()) + 1e-9  # fp32 sums of exact products
    assert bool(((frc.cpu().double() - want).abs() <= bound).all())


@pytest.mark.parametrize("M,D", [(2, 64), (5, 128), (31, 72), (32, 128), (33, 256), (64, 64), (100, 128),
                                 (127, 24), (128, 128)])
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("formula", ["additive", "multiplicative"])
@pytest.mark.parametrize("diagnostics", [True, False])
def test_same_bits_as_the_general_kernels(cuda, M, D, dt, formula, diagnostics):
    """The same matrix once alone (one kernel) and once inside one of 160 blocks (the
    general kernels) whose added keys score the minimum with every query: their
    column of Ahat is exactly 0, so they add exact zeros to every sum over keys and
    leave minimum and maximum as they are."""
    from cab_attention.kernels import compute_block_frc
    g = torch.Generator().manual_seed(M * 7 + D)
    big = 160
    q, k = (torch.randn((1, 2, big, D), generator=g) for _ in range(2))
    q[..., -1], k[..., -1] = 1.0, 0.0
    k[:, :, M - 1:] = 0.0          # key M - 1 is the first that scores the minimum,
    k[:, :, M - 1:, -1] = -512.0   # -512 * alpha, exact in every type
    q[:, :, M:] = q[:, :, :1]
    q, k = (x.to(DTYPES[dt]).to(cuda) for x in (q, k))
    kw = dict(lambda_redundancy=0.7, formula=formula, diagnostics=diagnostics)
    small = compute_block_frc(q[:, :, :M].contiguous(), k[:, :, :M].contiguous(), **kw)
    general = compute_block_frc(q, k, **kw)
    for a, b in zip(small, general):
        assert (a is None) == (b is None)
        if a is not None:
            assert torch.equal(a, b[:, :, :M, :M])
