"""The two forms of V in the 16-bit row-pair kernel: its rows through
transposing LDS reads (key blocks visited at most 48 times on average) and
tiles packed ahead (more, or token strides beyond 2^24): strides of V apart
from K's, ragged ends, both head dims, lists and dense calls on either side of
the line, against the oracle."""

import numpy as np
import pytest
import torch

from oracle import cab_oracle as O

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
ATOL = {"bf16": 2e-2, "fp16": 5e-3}


def _qkv(H, Hkv, Nq, Nk, D, dt, layout, cuda):
    g = torch.Generator().manual_seed(Nk + D)
    q = torch.randn((1, H, Nq, D), generator=g).to(DTYPES[dt])
    k = torch.randn((1, Hkv, Nk, D), generator=g).to(DTYPES[dt])
    v = torch.randn((1, Hkv, Nk, D), generator=g).to(DTYPES[dt])
    kd, vd = k.to(cuda), v.to(cuda)
    if layout == "v_wide":  # V inside a wider projection, K contiguous
        wide = torch.zeros((1, Nk, 3, Hkv, D), dtype=v.dtype, device=cuda)
        wide[:, :, 2] = vd.transpose(1, 2)
        vd = wide[:, :, 2].transpose(1, 2)
    elif layout == "k_wide":
        wide = torch.zeros((1, Nk, Hkv, D + 16), dtype=k.dtype, device=cuda)
        wide[..., :D] = kd.transpose(1, 2)
        kd = wide[..., :D].transpose(1, 2)
    f = [t.float().numpy() for t in (q, k, v)]
    return (q.to(cuda), kd, vd), f


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("layout", ["plain", "v_wide", "k_wide"])
@pytest.mark.parametrize("H,Hkv,Nq,Nk,causal", [
    (2, 2, 100, 100, True), (4, 2, 333, 333, True), (2, 1, 65, 1500, True),
    (2, 2, 700, 129, False),
    (4, 1, 1000, 1000, True),     # 4 x 16 x 1/2 = 32 visits: rows
    (4, 1, 2000, 1600, False),    # 128 visits: packed
])
def test_dense(cuda, H, Hkv, Nq, Nk, causal, dt, D, layout):
    from cab_attention.kernels import flash_attention
    qkv, f = _qkv(H, Hkv, Nq, Nk, D, dt, layout, cuda)
    out = flash_attention(*qkv, causal=causal)
    want, _, _ = O.dense_attention_scores(*(x.astype(np.float64) for x in f), causal=causal)
    assert np.abs(out.float().cpu().numpy() - want).max() <= ATOL[dt]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("layout", ["plain", "v_wide"])
@pytest.mark.parametrize("N,kmax,bs", [(1000, 5, 64), (64 * 49 + 1, 48, 64), (64 * 50, 49, 64),
                                       (1500, 3, 128)])
def test_lists(cuda, N, kmax, bs, dt, D, layout):
    from cab_attention.kernels import block_sparse_attention
    (q, k, v), f = _qkv(2, 2, N, N, D, dt, layout, cuda)
    M = (N + bs - 1) // bs
    rng = np.random.default_rng(N)
    idx = np.stack([np.sort(rng.permutation(M)[:kmax]) for _ in range(2 * M)])
    idx = idx.reshape(1, 2, M, kmax).astype(np.int32)
    cnt = np.full((1, 2, M), kmax, np.int32)
    cnt[..., ::4] = kmax - 1
    out = block_sparse_attention(q, k, v, torch.from_numpy(idx).to(cuda),
                                 torch.from_numpy(cnt).to(cuda), bs, causal=False)
    want = O.sparse_attention(*f, idx, cnt, bs, causal=False)
    assert np.abs(out.float().cpu().numpy() - want).max() <= ATOL[dt]


def test_v_rows_far_apart(cuda):
    """A V token stride beyond 2^24 elements takes the packed tiles."""
    from cab_attention.kernels import flash_attention
    Nk, D, step = 65, 64, (1 << 24) + 8
    (q, k, _), f = _qkv(1, 1, 70, Nk, D, "bf16", "plain", cuda)
    v = torch.from_numpy(f[2]).to(torch.bfloat16).to(cuda)
    far = torch.empty((Nk - 1) * step + D, dtype=torch.bfloat16, device=cuda)
    far = far.as_strided((1, 1, Nk, D), (step * Nk, step * Nk, step, 1))
    far.copy_(v)
    want, _, _ = O.dense_attention_scores(*(x.astype(np.float64) for x in f), causal=True)
    assert np.abs(flash_attention(q, k, far, causal=True).float().cpu().numpy() - want).max() <= ATOL["bf16"]


def _short_rows(x, stride):
    """Random values in x's shape, dtype and place, with a token stride below D:
    rows that overlap, or one row for all of them (stride 0)."""
    _, H, N, D = x.shape
    flat = torch.randn((1, H, (N - 1) * stride + D), generator=torch.Generator().manual_seed(N + D))
    flat = flat.to(x.dtype).to(x.device)
    return flat.as_strided((1, H, N, D), (flat.stride(0), flat.stride(1), stride, 1))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("stride", [0, 16, 56])
@pytest.mark.parametrize("which", ["q", "k", "v"])
@pytest.mark.parametrize("H,Hkv,Nq,Nk,causal", [
    (2, 2, 100, 100, True), (2, 1, 65, 1500, True), (2, 2, 40, 1300, False),
    (4, 1, 2000, 1600, False),  # 128 visits: packed
    (2, 2, 3, 400, True),       # few rows
])
def test_dense_rows_closer_than_their_length(cuda, H, Hkv, Nq, Nk, causal, which, stride, dt, D):
    """Token strides below D (an expanded row, overlapping windows) read the same
    rows as a contiguous copy: output and key totals."""
    from cab_attention.kernels import flash_attention_with_cumulative_scores
    qkv, _ = _qkv(H, Hkv, Nq, Nk, D, dt, "plain", cuda)
    at = "qkv".index(which)
    qkv = list(qkv)
    qkv[at] = _short_rows(qkv[at], stride)
    want, _, want_sc = O.dense_attention_scores(
        *(x.double().cpu().numpy() for x in qkv), causal=causal)
    out, sc = flash_attention_with_cumulative_scores(*qkv, causal=causal)
    assert np.abs(out.double().cpu().numpy() - want).max() <= ATOL[dt]
    np.testing.assert_allclose(sc.double().cpu().numpy(), want_sc, rtol=1e-2, atol=1e-4)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("which", ["q", "k", "v"])
@pytest.mark.parametrize("stride", [0, 16])
@pytest.mark.parametrize("N,kmax,bs", [(1000, 5, 64), (64 * 50, 49, 64), (1500, 3, 128), (700, 8, 32)])
def test_lists_rows_closer_than_their_length(cuda, N, kmax, bs, stride, which, D):
    from cab_attention.kernels import block_sparse_attention
    qkv, _ = _qkv(2, 2, N, N, D, "bf16", "plain", cuda)
    at = "qkv".index(which)
    qkv = list(qkv)
    qkv[at] = _short_rows(qkv[at], stride)
    M = (N + bs - 1) // bs
    rng = np.random.default_rng(N)
    idx = np.stack([np.sort(rng.permutation(M)[:kmax]) for _ in range(2 * M)])
    idx = idx.reshape(1, 2, M, kmax).astype(np.int32)
    cnt = np.full((1, 2, M), kmax, np.int32)
    out = block_sparse_attention(*qkv, torch.from_numpy(idx).to(cuda),
                                 torch.from_numpy(cnt).to(cuda), bs, causal=False)
    want = O.sparse_attention(*(x.float().cpu().numpy() for x in qkv), idx, cnt, bs, causal=False)
    assert np.abs(out.float().cpu().numpy() - want).max() <= ATOL["bf16"]
