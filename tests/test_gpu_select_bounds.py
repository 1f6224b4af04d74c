"""Selection without scores (fp64 scores of the columns that a 16-bit pass with
error bounds cannot rule out) against selection with scores (fp64 scores of
every column, held to the oracle elsewhere): the same positions, whatever the
keys; and against the oracle's own top-k of the returned scores."""
import numpy as np
import pytest
import torch

from oracle import selection as ref
from std_amd import ops
from tests.gpu_helpers import announce, cache_buffer, dev

pytestmark = pytest.mark.gpu


def _keys(kind, n_kv, P, gen):
    k = torch.randn(1, n_kv, P, 128, generator=gen)
    if kind == "wide":                                     # key norms over a factor of ten
        k *= torch.exp(torch.randn(1, n_kv, P, 1, generator=gen) * 0.7)
    elif kind == "dup":                                    # exact ties across the boundary
        k[:, :, P // 3:2 * (P // 3)] = k[:, :, :P // 3]
    elif kind == "equal":                                  # every score the same: more candidates than registers
        k[:] = k[:, :, :1]
    elif kind == "huge":                                   # no usable bound: every column is a candidate
        k *= 3e3
    elif kind == "tiny":
        k *= 1e-25
    elif kind == "overflow":                               # products past fp32, inside fp64
        k[:, :, 11] = 1e30
    elif kind == "nan":
        k[:, :, 7, 3] = float("nan")
        k[:, :, P // 2, 0] = float("inf")
    return k


def _check(q, k, text_start, vis, k_sel):
    args = (q.to(dev()), cache_buffer(k, k.shape[2] + 9), text_start, vis.to(dev()), k_sel)
    top, scores = ops.select_topk(*args, return_scores=True)
    alone = ops.select_topk(*args)
    torch.cuda.synchronize()
    assert torch.equal(top, alone)
    s = scores.cpu().numpy()
    if np.isfinite(s).all():
        v = vis.numpy()
        valid = (v >= 0) & (v < s.shape[1])
        for g in range(s.shape[0]):
            col = np.where(valid, s[g][np.clip(v, 0, s.shape[1] - 1)], 0.0)
            order = np.sort(np.argsort(-col, kind="stable")[:k_sel])
            np.testing.assert_array_equal(alone[g].cpu().numpy(), v[order])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("kind,n_q,n_kv,T,P,k_sel", [
    ("normal", 28, 4, 128, 3000, 700),
    ("normal", 28, 4, 23, 2049, 1),          # rows past a staging of 128 and a partial row tile
    ("normal", 7, 1, 5, 300, 295),           # every visual position
    ("wide", 32, 8, 37, 5000, 1500),
    ("dup", 28, 4, 20, 4001, 900),
    ("equal", 4, 2, 3, 9500, 4000),
    ("huge", 7, 1, 30, 1000, 100),
    ("tiny", 7, 1, 30, 1000, 100),
    ("nan", 8, 2, 16, 1500, 60),
    # from 2e6 scores on: the split row statistics, and the fp64 ones where they leave a head undecided
    ("normal", 28, 4, 40, 9001, 4000),
    ("normal", 7, 1, 700, 2100, 300),        # 4900 rows: part of the text inside the workgroups' rows
    ("wide", 28, 4, 100, 3000, 500),
    ("equal", 28, 4, 30, 3001, 700),
    ("huge", 28, 4, 64, 3000, 300),
    ("tiny", 28, 4, 64, 3000, 300),
    ("nan", 28, 4, 64, 3000, 300),
])
def test_positions_equal_the_full_pass(kind, n_q, n_kv, T, P, k_sel, dtype):
    announce(f"bounded selection {kind} {n_q}/{n_kv} T={T} P={P} k={k_sel} {dtype}")
    gen = torch.Generator().manual_seed(P + T)
    q = torch.randn(1, n_q, T, 128, generator=gen).to(dtype)
    k = _keys(kind, n_kv, P, gen).to(dtype)
    _check(q, k, P - T, torch.arange(P - T, dtype=torch.int32), k_sel)


@pytest.mark.parametrize("n_q,T,P", [(7, 9, 700), (28, 200, 1000)])
def test_overflowing_products(n_q, T, P):
    announce("bounded selection: products past fp32")
    gen = torch.Generator().manual_seed(3)
    q = (torch.randn(1, n_q, T, 128, generator=gen) * 1e12).to(torch.bfloat16)
    k = _keys("overflow", n_q // 7, P, gen).to(torch.bfloat16)
    _check(q, k, P - T, torch.arange(P - T, dtype=torch.int32), 50)


def test_close_scores_fall_back_to_fp64():
    """Key pairs that differ in one element's last bit by a little: the k-th and
    (k+1)-th scores are within the split statistics' error, and the fp64 ones decide."""
    announce("bounded selection: close scores")
    gen = torch.Generator().manual_seed(12)
    P, T = 4000, 40
    q = torch.randn(1, 28, T, 128, generator=gen).to(torch.bfloat16)
    q[..., 5] *= 2.0 ** -20
    k = torch.randn(1, 4, P, 128, generator=gen).to(torch.bfloat16)
    k[:, :, 2000:3900] = k[:, :, 50:1950]
    k[:, :, 2000:3900, 5] += 0.5                                  # moves a score by about 1e-7 of itself
    for k_sel in (101, 400, 901):
        _check(q, k, P - T, torch.arange(P - T, dtype=torch.int32), k_sel)


@pytest.mark.parametrize("T,P,k_sel", [(128, 9001, 3000), (20, 2500, 600)])
def test_more_candidates_than_one_tile_a_workgroup(T, P, k_sel):
    """Rows of 30 times the others' in one channel widen every bound: about a thousand
    candidates, more than 16 for each workgroup of a head (split and fp64 statistics)."""
    announce(f"bounded selection: many candidates T={T} P={P}")
    gen = torch.Generator().manual_seed(T)
    q = torch.randn(1, 28, T, 128, generator=gen)
    q[:, ::7, :, 5] *= 30 if P > 5000 else 100
    k = torch.randn(1, 4, P, 128, generator=gen)
    _check(q.to(torch.bfloat16), k.to(torch.bfloat16), P - T, torch.arange(P - T, dtype=torch.int32), k_sel)


def test_scattered_and_late_positions():
    """Gaps, positions inside the text rows (partly masked) and positions outside
    the prompt (score 0)."""
    announce("bounded selection: scattered, masked and invalid positions")
    gen = torch.Generator().manual_seed(4)
    P, T = 1800, 64
    q = torch.randn(1, 28, T, 128, generator=gen).to(torch.bfloat16)
    k = torch.randn(1, 4, P, 128, generator=gen).to(torch.bfloat16)
    vis = torch.cat([torch.arange(5, 1700, 3), torch.arange(1740, 1790, 2), torch.tensor([P + 3, P + 900])])
    _check(q, k, P - T, vis.to(torch.int32), 200)
    _check(q, k, P - T, vis.to(torch.int32), vis.numel())


def test_more_positions_than_one_emission_window():
    announce("bounded selection: 300000 positions")
    gen = torch.Generator().manual_seed(6)
    P = 300002
    q = torch.randn(1, 1, 2, 128, generator=gen).to(torch.bfloat16)
    k = torch.randn(1, 1, P, 128, generator=gen).to(torch.bfloat16)
    _check(q, k, P - 2, torch.arange(P - 2, dtype=torch.int32), 20000)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["fp16", "fp32"])
def test_probability_topk_with_ties(dtype):
    """The exact keys' candidates: mostly equal scores, and an infinite one."""
    announce(f"probability selection with ties {dtype}")
    gen = torch.Generator().manual_seed(8)
    n_kv, T, P, k_sel = 2, 3, 12001, 5000
    probs = torch.randint(0, 3, (1, 4, T, P), generator=gen).to(dtype) / 4
    probs[0, :, 0, 77] = float("inf")
    vis = torch.arange(P - T, dtype=torch.int32)
    top, scores = ops.select_topk_probs(probs.to(dev()), vis.to(dev()), k_sel, n_kv, return_scores=True)
    exp = ref.topk_positions(scores.cpu().numpy(), vis.numpy(), k_sel)
    np.testing.assert_array_equal(top.cpu().numpy(), exp)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("side", ["above", "below"])
def test_scores_beyond_the_first_parts(side, dtype):
    """Rows of 1024 in one channel, so that the first part of the split sees nothing of
    8 in the others and 16 in place of 9. Above: five keys score 1550 (log2), all of it
    beyond the first parts. Below: five keys score 4, of which the first parts see 1400."""
    announce(f"bounded selection: scores beyond the first parts, {side} {dtype}")
    gen = torch.Generator().manual_seed(21)
    P, T = 3000, 64
    q = torch.randn(1, 28, T, 128, generator=gen)
    k = torch.randn(1, 4, P, 128, generator=gen)
    if side == "above":
        q[:, :, ::2] = 8
        k[:, :, 100:600:100] = 12
    else:
        q[:, :, ::2, :100], q[:, :, ::2, 100:] = 9, 32
        k[..., 127] *= 0.05
        k[:, :, 100:600:100, :100], k[:, :, 100:600:100, 100:] = 16, -16.625
    q[:, :, ::2, 127] = 1024
    k[:, :, 100:600:100, 127] = 0
    _check(q.to(dtype), k.to(dtype), P - T, torch.arange(P - T, dtype=torch.int32), 300)


def test_scores_past_the_references_integers():
    """Powers of two, which the first part holds whole, with scores of 1e11: the
    reference, a float, steps by more than the exponents' range."""
    announce("bounded selection: scores of 1e11")
    gen = torch.Generator().manual_seed(22)
    P, T = 3000, 64
    q = torch.exp2(torch.randint(16, 19, (1, 28, T, 128), generator=gen).float())
    k = torch.exp2(torch.randint(16, 19, (1, 4, P, 128), generator=gen).float())
    k *= torch.randint(0, 2, k.shape, generator=gen) * 2 - 1
    _check(q.to(torch.bfloat16), k.to(torch.bfloat16), P - T, torch.arange(P - T, dtype=torch.int32), 300)


def test_fp16_elements_near_the_largest():
    """fp16 elements from 65280 on, whose first part would round to 65536."""
    announce("bounded selection: fp16 elements near the largest")
    gen = torch.Generator().manual_seed(23)
    P, T = 3000, 64
    q = torch.randn(1, 28, T, 128, generator=gen)
    q[..., 0] *= 1e-3
    k = torch.randn(1, 4, P, 128, generator=gen)
    k[:, :, 50:2500:50, 0] = torch.tensor([65280.0, 65472.0, 65504.0, -65504.0, 65248.0, -65280.0, 65312.0]).repeat(7)
    _check(q.half(), k.half(), P - T, torch.arange(P - T, dtype=torch.int32), 300)


@pytest.mark.parametrize("side", [1, -1])
@pytest.mark.parametrize("shift", [1e-10, 3e-11])
def test_tied_keys_next_to_a_close_one(side, shift):
    """Two equal keys straddle the k-th place below a third that scores 1e-5 more, and
    another key scores 1 + side x shift of theirs, closer than the split statistics'
    error: rows of one kind weigh the tied keys, rows of the other kind that one, on
    disjoint channels, so the two kinds' errors do not cancel."""
    announce(f"bounded selection: tied keys next to a close one {side} {shift}")
    gen = torch.Generator().manual_seed(24)
    n_kv, T, P, D = 4, 64, 9000, 128
    q = torch.zeros(1, n_kv, T, D)
    q[:, :, ::2, :60] = torch.randn(1, n_kv, T // 2, 60, generator=gen) * 4 + 20
    q[:, :, ::2, 60] = 2.0 ** -6
    q[:, :, 1::2, 64:123] = torch.randn(1, n_kv, T // 2, 59, generator=gen) + 1
    for c in range(5):                                     # fine channels of the second kind of row
        q[:, :, 1::2, 123 + c] = 2.0 ** (-4 - 8 * c)
    q = q.bfloat16()
    k = torch.randn(1, n_kv, P, D, generator=gen)
    k[..., :61] *= 0.03
    k[:, :, 20:60:10] = 0
    k[:, :, 20:50:10, :60] = 0.11
    k[:, :, 20, 60] = 0.02
    k = k.bfloat16()

    def gap(g):                                            # of keys 30 and 50, in 64 bits
        s = q[0, g].double() @ k[0, g].double().T / D ** 0.5
        s.masked_fill_(torch.arange(P)[None] > P - T + torch.arange(T)[:, None], float("-inf"))
        p = torch.softmax(s, -1).sum(0)
        return (p[50] / p[30] - 1 - side * shift).item()

    for g in range(n_kv):
        # the close key: along the second kind's mean, then channel by channel nearer
        for c, reach in [(slice(64, 123), 4.0)] + [(c, 64.0) for c in range(123, 128)]:
            lo, hi, best = -reach, reach, (9.0, 0.0)
            for _ in range(16):
                mid = (lo + hi) / 2
                k[0, g, 50, c] = mid
                x = gap(g)
                best = min(best, (abs(x), mid))
                lo, hi = (mid, hi) if x < 0 else (lo, mid)
            k[0, g, 50, c] = best[1]
        assert abs(gap(g)) < shift / 4
    vis = torch.arange(P - T, dtype=torch.int32)
    scores = ops.select_topk(q.to(dev()), k.to(dev()), P - T, vis.to(dev()), 4, return_scores=True)[1].cpu()
    above = {int((scores[g, :P - T] > scores[g, 20]).sum()) for g in range(n_kv)}
    for k_sel in sorted({a + i for a in above for i in (1, 2, 3)}):
        _check(q, k, P - T, vis, k_sel)


@pytest.mark.parametrize("P", [2000, 16000])               # fp64 statistics; split ones, which leave it undecided
def test_scores_equal_but_for_rounding(P):
    """Pairs of keys whose scores are the same sums of the same terms in another order:
    they differ in their last bits, by the order of the additions alone."""
    announce(f"bounded selection: scores equal but for rounding, {P} keys")
    gen = torch.Generator().manual_seed(25)
    T, n = 40, (P - 40) // 2
    q = torch.randn(1, 8, T, 128, generator=gen)
    q[:, 1::2] = q[:, ::2].flip(-1)
    k = torch.randn(1, 2, P, 128, generator=gen)
    k[:, :, n:2 * n] = k[:, :, :n].flip(-1)
    k[:, :, 2 * n:, 64:] = k[:, :, 2 * n:, :64].flip(-1)
    for k_sel in range(101, 500, 26):
        _check(q.bfloat16(), k.bfloat16(), P - T, torch.arange(2 * n, dtype=torch.int32), k_sel)
