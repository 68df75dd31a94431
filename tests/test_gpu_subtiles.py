"""Block sizes below 64: lists without repeats are merged through one mask per
64-token tile, quadrants of a tile without kept blocks are skipped, and key
ranges beyond the merge's 4096 tiles take the list-order merge. Outputs
against the oracle on sampled query blocks, both head dims and all types."""

import numpy as np
import pytest
import torch

from oracle import cab_oracle as O

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ATOL = {"bf16": 2e-2, "fp16": 5e-3, "fp32": 1e-3}  # as for the executor's other tests


def _run(cuda, N, D, bs, dt, k, causal, seed):
    from cab_attention.kernels import block_sparse_attention
    H, Mb = 2, (N + bs - 1) // bs
    rng = np.random.default_rng(seed)
    # k distinct blocks a row in random order (some past the causal limit),
    # the last slot of every third row empty; row 1 without any.
    idx = np.stack([rng.permutation(Mb)[:k] if Mb < 4096 else
                    np.unique(rng.integers(0, Mb, 4 * k))[:: -1][:k]
                    for _ in range(H * Mb)]).reshape(1, H, Mb, k).astype(np.int32)
    cnt = np.full((1, H, Mb), k, np.int32)
    cnt[..., ::3] = k - 1
    cnt[..., 1] = 0
    g = torch.Generator().manual_seed(seed)
    q, kk, v = (torch.randn((1, H, N, D), generator=g).to(DTYPES[dt]) for _ in range(3))
    out = block_sparse_attention(q.to(cuda), kk.to(cuda), v.to(cuda), torch.from_numpy(idx).to(cuda),
                                 torch.from_numpy(cnt).to(cuda), bs, causal=causal)
    rows = sorted({0, 1, 2, Mb // 2, Mb // 2 + 1, Mb - 2, Mb - 1})
    f = [t.float().numpy() for t in (q, kk, v)]
    want = O.sparse_attention(*f, idx, cnt, bs, causal=causal, query_blocks=rows)
    got = out.float().cpu().numpy()
    for i in rows:
        sl = slice(bs * i, min(bs * i + bs, N))
        assert np.abs(got[:, :, sl] - want[:, :, sl]).max() <= ATOL[dt], f"row {i}"


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("causal", [False, True])
def test_lists_without_repeats(cuda, bs, dt, D, causal):
    _run(cuda, 64 * 9 + 5, D, bs, dt, 4, causal, 7 * bs + D)


def test_more_tiles_than_the_merge_holds(cuda):
    _run(cuda, 64 * 4097, 64, 32, "bf16", 3, False, 3)
