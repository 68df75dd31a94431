"""Dense attention for few query rows (decode steps, short chunks) with the
key totals in the same call: cab_flash_attn_scores_fwd at the edges of the
key split (32-key steps, four per workgroup), of the row tiles (16 and 32
rows per K / V head, and 33, which runs the general kernels), of the general
kernels' own split over the keys, and of the running totals (none, shorter,
as long as the keys), against the float64 oracle; and cab_flash_attn_fwd with
a workspace the partials do not fit."""

import math

import numpy as np
import pytest
import torch

from oracle import cab_oracle as O

from cab_attention import _native as nat

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
# As for the other dense kernels: rounding of P and of the output for the
# 16-bit types, split bf16 operands (2^-16 a product) for fp32.
ATOL = {"bf16": 2e-2, "fp16": 5e-3, "fp32": 1e-3}
LSE_ATOL = {"bf16": 2e-3, "fp16": 1e-3, "fp32": 1e-3}


def seeded(shape, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g, dtype=torch.float32).to(dtype)


def np64(t):
    return t.detach().double().cpu().numpy()


CASES = [  # (B, H, H_kv, N_q, N_k)
    (1, 4, 4, 1, 1),
    (2, 4, 1, 1, 31),
    (1, 8, 2, 1, 32),
    (1, 2, 2, 1, 33),
    (3, 14, 2, 1, 129),      # 7 rows; one key past a workgroup's four steps
    (1, 4, 4, 16, 500),      # a full row tile
    (1, 4, 4, 17, 1025),     # one row into the second; one key past a totals chunk
    (2, 8, 2, 8, 1000),      # 32 rows
    (1, 32, 4, 3, 4099),     # 24 rows: the second tile half empty
    (1, 3, 1, 11, 700),      # 33 rows: the general kernels
    (1, 2, 1, 16, 7),        # more queries than keys (causal: the first see none)
    (1, 4, 2, 33, 1250),     # general kernels, one block short of two parts
    (1, 4, 2, 33, 1281),     # keys split in two, one key in the last block
    (1, 4, 4, 130, 2100),    # three parts, the last one past the first queries' keys
    (1, 2, 2, 40, 6000),     # eight parts, the most
]


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,H,Hkv,Nq,Nk", CASES)
def test_rows_and_totals(cuda, B, H, Hkv, Nq, Nk, causal, dt, D):
    from cab_attention.kernels import flash_attention, flash_attention_with_cumulative_scores
    # K and V as views of [B, N, H_kv, D] rows, as a projection leaves them.
    q = seeded((B, H, Nq, D), 1, DTYPES[dt]).to(cuda)
    k = seeded((B, Nk, Hkv, D), 2, DTYPES[dt]).to(cuda).transpose(1, 2)
    v = seeded((B, Nk, Hkv, D), 3, DTYPES[dt]).to(cuda).transpose(1, 2)
    w_out, w_lse, w_sc = O.dense_attention_scores(np64(q), np64(k), np64(v), causal=causal)
    out, lse = flash_attention(q, k, v, causal=causal, return_lse=True)
    fin = np.isfinite(w_lse)
    assert np.array_equal(np.isfinite(np64(lse)), fin)
    np.testing.assert_allclose(np64(lse)[fin], w_lse[fin], atol=LSE_ATOL[dt], rtol=1e-4)
    assert np.abs(np64(out) - w_out).max() <= ATOL[dt]
    for n_old in sorted({0, Nk - 1, Nk}):
        old = None if n_old == 0 else torch.rand((B, H, n_old), device=cuda)
        base = np.zeros((B, H, Nk))
        if old is not None:
            base[..., :n_old] = np64(old)
        out2, sc = flash_attention_with_cumulative_scores(q, k, v, old, causal=causal)
        assert torch.equal(out2, out)
        assert (sc is old) == (n_old == Nk and old is not None)
        # This call's part of the totals: lse sums P rounded to a 16-bit type (2^-9
        # relative per query at most; fp32: split products, 2^-16), and the sum
        # with the old totals (below 1) is rounded to fp32.
        np.testing.assert_allclose(np64(sc) - base, w_sc, rtol=1e-4 if dt == "fp32" else 5e-3,
                                   atol=2.0 ** -22)


def test_growing_maxima(cuda):
    """Scores that grow along the keys (every step raises the running maximum)."""
    from cab_attention.kernels import flash_attention
    B, H, Nq, Nk, D = 1, 4, 3, 700, 128
    q = seeded((B, H, Nq, D), 1, torch.bfloat16)
    k = seeded((B, H, Nk, D), 2, torch.bfloat16)
    v = seeded((B, H, Nk, D), 3, torch.bfloat16)
    k = k + (q.float().mean(2, keepdim=True) * torch.linspace(0, 4, Nk)[:, None]).to(k.dtype)
    w_out, w_lse, _ = O.dense_attention_scores(np64(q), np64(k), np64(v), causal=True)
    out, lse = flash_attention(q.to(cuda), k.to(cuda), v.to(cuda), causal=True, return_lse=True)
    assert np.abs(np64(out) - w_out).max() <= ATOL["bf16"]
    np.testing.assert_allclose(np64(lse), w_lse, atol=LSE_ATOL["bf16"], rtol=1e-4)


def test_shorter_totals_carry_their_gradient(cuda):
    """Totals that are extended to new keys stay in the graph they come from (the
    call's own totals have none)."""
    from cab_attention.kernels import flash_attention_with_cumulative_scores
    q, k, v = (seeded((1, 2, n, 64), n, torch.bfloat16).to(cuda) for n in (3, 40, 40))
    old = torch.rand((1, 2, 33), device=cuda, requires_grad=True)
    _, sc = flash_attention_with_cumulative_scores(q, k, v, old * 2.0)
    _, plain = flash_attention_with_cumulative_scores(q, k, v, (old * 2.0).detach())
    assert torch.equal(sc.detach(), plain)
    sc.square().sum().backward()
    torch.testing.assert_close(old.grad, 4.0 * plain[..., :33])
    neg = torch._neg_view(old.detach())
    _, sc = flash_attention_with_cumulative_scores(q, k, v, neg)
    _, plain = flash_attention_with_cumulative_scores(q, k, v, -old.detach())
    assert torch.equal(sc, plain)


@pytest.mark.parametrize("dt", ["bf16", "fp32"])
def test_flash_fwd_workspace_decides_the_path(cuda, dt):
    """cab_flash_attn_fwd takes its documented workspace whatever path runs: for
    16-bit inputs the partials of 32 rows over 64 keys are larger than the
    packed block, so the general kernels run there; with a larger workspace
    the few-row ones do."""
    lib = nat.load()
    B, H, Hkv, Nq, Nk, D = 1, 32, 1, 1, 64, 128
    q = seeded((B, H, Nq, D), 5, DTYPES[dt]).to(cuda)
    k = seeded((B, Hkv, Nk, D), 6, DTYPES[dt]).to(cuda)
    v = seeded((B, Hkv, Nk, D), 7, DTYPES[dt]).to(cuda)
    w_out, w_lse, _ = O.dense_attention_scores(np64(q), np64(k), np64(v), causal=True)
    code = nat.dtype_code(q)
    need = int(lib.cab_flash_attn_workspace_bytes(code, B, Hkv, Nk, D))
    for size in (need, need + (1 << 20)):
        out = torch.empty_like(q)
        lse = torch.empty((B, H, Nq), device=cuda)
        ws = torch.empty(size, dtype=torch.uint8, device=cuda)
        st = lib.cab_flash_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), code, B, H, Hkv, Nq,
                                    Nk, D, nat.strides4(q), nat.strides4(k), nat.strides4(v),
                                    nat.strides4(out), 1.0 / math.sqrt(D), 1, out.data_ptr(),
                                    lse.data_ptr(), ws.data_ptr(), ws.numel(),
                                    torch.cuda.current_stream(cuda).cuda_stream)
        nat.check("cab_flash_attn_fwd", st)
        assert np.abs(np64(out) - w_out).max() <= ATOL[dt]
        np.testing.assert_allclose(np64(lse), w_lse, atol=LSE_ATOL[dt], rtol=1e-4)
