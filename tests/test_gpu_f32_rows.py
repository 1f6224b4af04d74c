"""fp32 attention at the edges of its row pairs (32 rows a workgroup), its waves'
16 keys and its tiles, with and without the fused append, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import attention as ref
from std_amd import ops
from tests.gpu_helpers import announce, cache_buffer, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_q,n_kv,q_len,kv_len", [
    (n_q, n_kv, q_len, kv_len)
    for n_q, n_kv, q_len in [(7, 1, 1), (16, 1, 1), (17 * 2, 2, 1), (16, 1, 2), (33, 3, 3), (28, 4, 10), (8, 1, 12)]
    for kv_len in [1, 15, 16, 17, 64, 65, 80, 81, 700] if kv_len >= q_len])
def test_f32_rows(n_q, n_kv, q_len, kv_len):
    announce(f"fp32 rows {n_q}/{n_kv} q={q_len} kv={kv_len}")
    gen = torch.Generator().manual_seed(kv_len * 100 + q_len)
    q = torch.randn(1, n_q, q_len, 128, generator=gen)
    q[:, :, -1] *= 5                                              # a peaked row: the maximum rises late
    k, v = (torch.randn(1, n_kv, kv_len, 128, generator=gen) for _ in "kv")
    kb, vb = cache_buffer(k, kv_len + 21), cache_buffer(v, kv_len + 21)
    exp = ref.verify_attention(q, k, v)
    # A score's error e changes an output by at most 2 e max|v|, |v| < 5 here, whatever
    # the output itself is. A dot product of 128 terms rounds at most 34 times along a
    # chain, at 2^-24 of partial sums that stay below 30 (150 in the peaked row), and is
    # divided by sqrt(128): e < 34 x 6e-8 x 30 / 11.3 = 5.4e-6 at worst, a fifth of it for
    # rounding errors of random sign, and five times that in the peaked row.
    def close(got):
        got = got.cpu().numpy()
        np.testing.assert_allclose(got[:, :, :-1], exp[:, :, :-1], rtol=2e-5, atol=1e-5)
        np.testing.assert_allclose(got[:, :, -1], exp[:, :, -1], rtol=2e-5, atol=5e-5)

    out = ops.verify_attention(q.to(dev()), kb[:, :, :kv_len], vb[:, :, :kv_len])
    close(out)
    first = kv_len - q_len
    kb[:, :, first:], vb[:, :, first:] = float("nan"), float("nan")   # the append brings the last rows
    nk, nv = k[:, :, first:].to(dev()), v[:, :, first:].to(dev())
    again = ops.verify_attention_append(q.to(dev()), kb, vb, nk, nv, kv_len)
    assert torch.equal(out, again)
    assert torch.equal(kb[:, :, first:kv_len], nk) and torch.equal(vb[:, :, first:kv_len], nv)
    assert torch.isnan(kb[:, :, kv_len:]).all()


@pytest.mark.parametrize("kv_len", [3, 70, 700])
def test_f32_infinite_last_value(kv_len):
    """The last key's value infinite in two columns, off the tile: infinite there for the
    row that sees it, untouched elsewhere (rows past the cache's last are not values)."""
    announce(f"fp32 infinite last value kv={kv_len}")
    gen = torch.Generator().manual_seed(kv_len)
    q = torch.randn(1, 7, 1, 128, generator=gen)
    k, v = (torch.randn(1, 1, kv_len, 128, generator=gen) for _ in "kv")
    exp = torch.from_numpy(ref.verify_attention(q, k, v)).float()
    v[0, 0, -1, 5], v[0, 0, -1, 77] = float("inf"), float("-inf")
    exp[..., 5], exp[..., 77] = float("inf"), float("-inf")
    out = ops.gqa_decode(q.to(dev()), cache_buffer(k, kv_len + 9)[:, :, :kv_len],
                         cache_buffer(v, kv_len + 9)[:, :, :kv_len]).cpu()
    torch.testing.assert_close(out, exp, rtol=2e-5, atol=5e-5)
