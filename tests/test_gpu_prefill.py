"""GPU parity of the prompt attention (ops.prefill_attention) against the
oracle's causal attention in fp64."""
import pytest
import torch

from oracle import attention as ref
from std_amd import ops
from tests.gpu_helpers import announce, dev

pytestmark = pytest.mark.gpu

# An output row is a weighted mean of the values: its error is the final
# rounding to the element type (2^-9 and 2^-12 relative at most, about 0.58 of
# half that in the 2-norm) plus fp32 terms 100 times smaller.
REL = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("n_q,n_kv,n,past", [
    (28, 4, 1, 0),        # one row, one key
    (28, 4, 14, 63),      # the smallest prompt past the decode rows; the last key starts a tile
    (7, 1, 32, 32),       # one row tile per head, keys ending on a tile
    (7, 1, 33, 31),       # a row tile of one row
    (16, 2, 64, 0),       # whole workgroups, no past
    (4, 4, 257, 0),       # no sharing: a workgroup spans 256 positions and four key tiles of the diagonal
    (28, 4, 128, 1500),   # a text suffix: split keys and the merge
    (32, 8, 300, 77),
    (28, 4, 20, 513),     # eight key tiles and one key: two splits at most
    (16, 1, 600, 5),      # the largest group
])
def test_prefill_attention_matches_oracle(n_q, n_kv, n, past, dtype):
    announce(f"prefill attention {n_q}/{n_kv} n={n} past={past} {dtype}")
    gen = torch.Generator().manual_seed(n * 1000 + past)
    kv = past + n
    q = torch.randn(1, n, n_q, 128, generator=gen).to(dtype)
    q[:, n // 2:] *= 4                                        # peaked rows raise the running maximum late
    k, v = (torch.randn(1, n_kv, kv, 128, generator=gen).to(dtype) for _ in "kv")
    kb, vb = (torch.full((1, n_kv, kv + 5, 128), float("nan"), dtype=dtype, device=dev()) for _ in "kv")
    kb[:, :, :kv], vb[:, :, :kv] = k.to(dev()), v.to(dev())
    exp = torch.from_numpy(ref.verify_attention(q.transpose(1, 2), k, v))
    for query in (q.to(dev()).transpose(1, 2), q.transpose(1, 2).contiguous().to(dev())):   # both query layouts
        out = ops.prefill_attention(query, kb, vb, kv)
        assert out.shape == query.shape and out.transpose(1, 2).is_contiguous()
        got = out.cpu().double()
        assert torch.isfinite(got).all()
        assert ((got - exp).norm() / exp.norm()).item() <= REL[dtype]
        assert torch.equal(out, ops.prefill_attention(query, kb, vb, kv))                   # and deterministic


def test_prefill_attention_extreme_scores():
    """Scores far from zero in both directions: a first tile of very low
    scores, then higher ones, and a key that takes all the weight."""
    announce("prefill attention extreme scores")
    dtype = torch.bfloat16
    gen = torch.Generator().manual_seed(5)
    n, n_q, n_kv = 200, 7, 1
    q = torch.randn(1, n_q, n, 128, generator=gen).abs().to(dtype)
    k = torch.randn(1, n_kv, n, 128, generator=gen)
    k[:, :, :64] -= 100.0
    k[:, :, 150] += 30.0
    k, v = k.to(dtype), torch.randn(1, n_kv, n, 128, generator=gen).to(dtype)
    out = ops.prefill_attention(q.to(dev()), k.to(dev()), v.to(dev()), n).cpu().double()
    exp = torch.from_numpy(ref.verify_attention(q, k, v))
    assert torch.isfinite(out).all()
    # scores of magnitude 1e4 carry an fp32 rounding of about 1e-3, which is a
    # probability's relative error; the rest is the output's rounding
    assert ((out - exp).norm() / exp.norm()).item() <= 2.0 ** -9 + 2e-3


def test_prefill_attention_rejects():
    q = torch.zeros(1, 4, 8, 128, dtype=torch.bfloat16, device=dev())
    k = torch.zeros(1, 4, 16, 128, dtype=torch.bfloat16, device=dev())
    with pytest.raises(ValueError):
        ops.prefill_attention(q, k, k, 17)
    with pytest.raises(ValueError):
        ops.prefill_attention(q, k, k, 7)
    with pytest.raises(RuntimeError):
        ops.prefill_attention(q, k, k, 16, scale=-1.0)
    with pytest.raises(RuntimeError):
        ops.prefill_attention(q.float(), k.float(), k.float(), 16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("n,past,peak", [(1500, 0, 1.0), (128, 6000, 1.0), (700, 90, 4.0)])
def test_prefill_attention_is_as_close_as_fp32(n, past, peak, dtype):
    """Probabilities and sums are held to 32 bits: no larger share of the outputs than
    with fp32 matrix products is another number than the rounded 64-bit value. (An output
    is misrounded where its error before rounding crosses a rounding boundary, so the
    share is proportional to that error; 8e5 outputs and more, a share of 4e-4 and more
    is known to 3 standard deviations of 17 %.)"""
    announce(f"prefill attention against fp32 products n={n} past={past} {dtype}")
    gen = torch.Generator().manual_seed(n)
    kv, n_q, n_kv = past + n, 14, 2
    q = (torch.randn(n_q, n, 128, generator=gen) * peak).to(dtype).to(dev())
    k, v = (torch.randn(n_kv, kv, 128, generator=gen).to(dtype).to(dev()) for _ in "kv")
    got = ops.prefill_attention(q[None], k[None], v[None], kv)[0]
    hidden = torch.arange(kv, device=dev())[None] > past + torch.arange(n, device=dev())[:, None]
    wrong = {"kernel": 0, "fp32": 0}
    for h in range(n_q):
        def products(t):
            s = q[h].to(t) @ k[h // 7].to(t).t().contiguous() / 128 ** 0.5
            return torch.softmax(s.masked_fill_(hidden, float("-inf")), -1) @ v[h // 7].to(t)
        exact = products(torch.float64).float().to(dtype)
        wrong["fp32"] += (products(torch.float32).to(dtype) != exact).sum().item()
        wrong["kernel"] += (got[h] != exact).sum().item()
    assert wrong["kernel"] <= 1.2 * wrong["fp32"], wrong
