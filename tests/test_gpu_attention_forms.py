"""The attention wrappers' short form check: what it does not take goes through
every check and gives the same result or the same error; and any scale."""
import numpy as np
import pytest
import torch

from oracle import attention as ref
from std_amd import ops
from tests.gpu_helpers import announce, assert_close, cache_buffer, dev

pytestmark = pytest.mark.gpu


def _case(q_len=1):
    gen = torch.Generator().manual_seed(11)
    mk = lambda *s: torch.randn(*s, generator=gen).to(torch.bfloat16).to(dev())
    return mk(1, 14, q_len, 128), mk(1, 2, 96, 128), mk(1, 2, 96, 128), mk(1, 2, q_len, 128), mk(1, 2, q_len, 128)


def test_forms_give_the_same_result():
    announce("attention forms")
    q, k, v, nk, nv = _case()
    fn = lambda nk, nv, n, **kw: ops.gqa_decode_append(q, k.clone(), v.clone(), nk, nv, n, **kw)
    exp = fn(nk, nv, 70)
    out = torch.empty_like(q)
    assert fn(nk, nv, 70, out=out) is out and torch.equal(out, exp)
    assert torch.equal(fn(nk, nv, np.int64(70)), exp)
    odd = nv.as_strided(nv.shape, (7, 128, 999, 1))               # another stride of size-1 dimensions
    assert torch.equal(fn(nk, odd, 70), exp)
    wide = torch.empty(1, 2, 128, 128, dtype=v.dtype, device=dev())
    wide[:, :, :96] = v
    assert torch.equal(ops.gqa_decode(q, k, wide[:, :, :96]), ops.gqa_decode(q, k, v))   # its own head stride


@pytest.mark.parametrize("change,error", [
    (lambda a: a.update(nv=a["nv"].float()), TypeError),
    (lambda a: a.update(v=a["v"].float()), TypeError),
    (lambda a: a.update(nk=a["nk"][:, :1]), ValueError),
    (lambda a: a.update(n=97), ValueError),
    (lambda a: a.update(n=0), ValueError),
    (lambda a: a.update(v=a["v"][:, :, :90]), ValueError),
    (lambda a: a.update(k=a["k"][:, :, ::2], v=a["v"][:, :, ::2]), ValueError),
    (lambda a: a.update(q=a["q"][:, :13]), ValueError),
    (lambda a: a.update(q=a["q"].transpose(1, 3)), ValueError),
    (lambda a: a.update(k=a["k"].cpu()), RuntimeError),
    (lambda a: a.update(nv=a["nv"].transpose(1, 3).contiguous().transpose(1, 3)), ValueError),
])
def test_forms_refused(change, error):
    a = dict(zip(("q", "k", "v", "nk", "nv"), _case()), n=70)
    change(a)
    with pytest.raises(error):
        ops.gqa_decode_append(a["q"], a["k"], a["v"], a["nk"], a["nv"], a["n"])


def test_streams_have_their_own_workspace():
    announce("attention on a second stream")
    q, k, v, _, _ = _case(5)
    exp = ops.verify_attention(q, k, v)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = ops.verify_attention(q, k, v)
        assert ops._stream(q.device) == side.cuda_stream
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, exp)
    assert ops._stream(q.device) == torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("scale", [0.0, -0.125])
@pytest.mark.parametrize("q_len,kv_len", [(1, 70), (1, 300), (5, 70), (10, 333)])
def test_any_scale(q_len, kv_len, scale, dtype):
    """Scale 0 (the mean of the values seen) and a negative one, off the tile: the mask
    and the running maximum are those of the scaled scores."""
    announce(f"attention scale {scale} q={q_len} kv={kv_len} {dtype}")
    gen = torch.Generator().manual_seed(q_len + kv_len)
    q = torch.randn(1, 14, q_len, 128, generator=gen).to(dtype)
    k, v = (torch.randn(1, 2, kv_len, 128, generator=gen).to(dtype) for _ in "kv")
    exp = ref.verify_attention(q, k, v, scale=scale)
    kb, vb = cache_buffer(k, kv_len + 30), cache_buffer(v, kv_len + 30)
    assert_close(ops.verify_attention(q.to(dev()), kb[:, :, :kv_len], vb[:, :, :kv_len], scale=scale), exp, dtype)
    new = [x[:, :, kv_len - q_len:].to(dev()) for x in (k, v)]
    assert_close(ops.verify_attention_append(q.to(dev()), kb, vb, *new, kv_len, scale=scale), exp, dtype)
    if q_len == 1:
        assert_close(ops.gqa_decode(q.to(dev()), kb[:, :, :kv_len], vb[:, :, :kv_len], scale=scale), exp, dtype)
