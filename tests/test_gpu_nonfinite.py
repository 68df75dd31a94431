"""NaN and infinities in q, k and v of the dense calls: the outputs and key
totals that are not finite are those a float64 softmax has, whichever kernels
run (few rows, the key blocks split into two and into four parts, unsplit)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ROUTES = [  # (H, H_kv, N_q, N_k)
    (4, 2, 3, 200),     # few rows
    (8, 2, 1, 700),
    (4, 4, 24, 1100),
    (2, 2, 33, 1281),   # key blocks in two parts (16-bit types), the last holds one key
    (4, 2, 100, 2700),  # four parts
    (4, 2, 100, 300),   # one part
]


def softmax_reference(q, k, v, causal):
    """Output and key totals in float64; a masked key's V is multiplied by nothing."""
    H, Hkv, Nq, Nk = q.shape[1], k.shape[1], q.shape[2], k.shape[2]
    q, k, v = (t.double() for t in (q, k, v))
    k, v = (t.repeat_interleave(H // Hkv, 1) for t in (k, v))
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / q.shape[-1] ** 0.5
    gone = torch.zeros((Nq, Nk), dtype=torch.bool)
    if causal:
        gone = torch.arange(Nk)[None, :] > torch.arange(Nq)[:, None] + Nk - Nq
    p = torch.softmax(s.masked_fill(gone, -torch.inf), -1).masked_fill(gone, 0.0)
    return torch.matmul(p, v), p.sum(2)


@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("H,Hkv,Nq,Nk", ROUTES)
@pytest.mark.parametrize("where", ["q_nan", "k_nan", "k_nan_last", "k_inf", "v_nan", "v_inf"])
def test_nonfinite_inputs(cuda, where, H, Hkv, Nq, Nk, causal, dt):
    from cab_attention.kernels import flash_attention_with_cumulative_scores
    if dt == "fp32" and where.endswith("inf"):
        pytest.skip("fp32 operands are split into bf16 halves: inf - inf is NaN there")
    g = torch.Generator().manual_seed(Nk)
    D = 64
    q, k, v = (torch.randn((1, h, n, D), generator=g).to(DTYPES[dt])
               for h, n in ((H, Nq), (Hkv, Nk), (Hkv, Nk)))
    if where == "q_nan":
        q[0, 1, Nq // 2, 5] = torch.nan
    elif where == "k_nan":
        k[0, 0, 70, 3] = torch.nan
    elif where == "k_nan_last":  # causal: the last query alone sees it
        k[0, 0, -1, 3] = torch.nan
    elif where == "k_inf":  # scores of +inf (NaN rows) and of -inf (no weight)
        k[0, 0, 70, 3] = torch.inf
    elif where == "v_nan":
        v[0, 0, 5, 3] = torch.nan
    else:
        v[0, 0, 5, 3] = torch.inf
    want, want_sc = softmax_reference(q, k, v, causal)
    out, sc = flash_attention_with_cumulative_scores(q.to(cuda), k.to(cuda), v.to(cuda),
                                                     causal=causal)
    fin, fin_sc = torch.isfinite(want), torch.isfinite(want_sc)
    assert not bool(fin.all()), "the case has to reach an output"
    assert torch.equal(torch.isfinite(out.cpu()), fin)
    assert torch.equal(torch.isfinite(sc.cpu()), fin_sc)
    atol = {"bf16": 2e-2, "fp16": 5e-3, "fp32": 1e-3}[dt]
    assert float((out.cpu().double() - want)[fin].abs().max()) <= atol
    # (P is summed as rounded to the data type: 2^-9 relative per query)
    torch.testing.assert_close(sc.cpu().double()[fin_sc], want_sc[fin_sc], rtol=5e-3, atol=1e-4)
