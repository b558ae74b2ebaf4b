"""The prompt pass's attention kernel (hqq_attention_rows) against softmax attention in 64 bits on the same fp16 inputs.

Tolerance: the kernel's sums are fp32; what it rounds is a probability of at most 1 to fp16 (2^-11 of it, or 2^-25 below
fp16's normal range) and the output to fp16, so an element is off by at most 2^-11 (sum_k p_k |v_k| + |out|) + 2^-25
sum_k |v_k| / sum and the fp32 parts, far below; twice that bound is allowed."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(tokens, start, heads, kv, hd, room=3, seed=0, spread=1.0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    q = (torch.randn((tokens, heads, hd), device="cuda", generator=gen) * spread).half()
    ck, cv = (torch.randn((kv, start + tokens + room, hd), device="cuda", generator=gen).half() for _ in range(2))
    ck[:, start + tokens:], cv[:, start + tokens:] = float("nan"), float("nan")  # positions no token may read
    return q, ck, cv


def _reference(q, ck, cv, start):
    tokens, heads, hd = q.shape
    kv, total = ck.shape[0], start + tokens
    k, v = ck[:, :total].double().cpu(), cv[:, :total].double().cpu()
    qd = q.double().cpu()
    later = torch.arange(total)[None, :] > start + torch.arange(tokens)[:, None]
    out, bound = torch.empty((tokens, heads, hd), dtype=torch.float64), torch.empty((tokens, heads, hd), dtype=torch.float64)
    for h in range(heads):
        j = h // (heads // kv)
        p = torch.softmax((qd[:, h] @ k[j].T / hd ** 0.5).masked_fill(later, float("-inf")), dim=-1)
        out[:, h] = p @ v[j]
        bound[:, h] = 2.0 ** -11 * (p @ v[j].abs() + out[:, h].abs()) + 2.0 ** -25 * (~later).double() @ v[j].abs()
    return out.reshape(tokens, -1), bound.reshape(tokens, -1)


@pytest.mark.parametrize("tokens,start", [(1, 0), (2, 0), (15, 0), (16, 1), (17, 63), (33, 64), (64, 0), (65, 100), (127, 1),
                                          (130, 0), (257, 31)])
@pytest.mark.parametrize("heads,kv,hd", [(32, 8, 128), (4, 2, 64), (3, 1, 128), (2, 2, 64)])
def test_attention_rows(tokens, start, heads, kv, hd):
    from mixtral_offloading_amd import hip_kernels
    q, ck, cv = _case(tokens, start, heads, kv, hd, seed=tokens + start)
    want, bound = _reference(q, ck, cv, start)
    got = hip_kernels.attention_rows(q, ck, cv, start).double().cpu()
    assert ((got - want).abs() <= 2 * bound).all()


@pytest.mark.parametrize("tokens,spread,hd", [(2048, 1.0, 128), (2100, 6.0, 128), (2050, 1.0, 64)])
def test_attention_rows_two_tiles_a_wave(tokens, spread, hd):
    """From 512 blocks a wave takes two query tiles (32 heads on 8 key/value heads: 2017 tokens)."""
    from mixtral_offloading_amd import hip_kernels
    q, ck, cv = _case(tokens, 5, 32, 8, hd, seed=tokens, spread=spread)
    want, bound = _reference(q, ck, cv, 5)
    got = hip_kernels.attention_rows(q, ck, cv, 5).double().cpu()
    assert ((got - want).abs() <= 2 * bound).all()


def _parts(tokens, start, heads, kv, hd):
    """Parts the positions of a call are split into, from the size of the scratch it asks for."""
    from mixtral_offloading_amd import _lib
    return max(1, _lib.lib.hqq_attention_rows_workspace_bytes(start, tokens, heads, kv, hd) // (4 * (hd + 2) * heads * tokens))


# few tokens behind many positions, each with more than one part; the last part short or one position long, blocks that
# see less than the last part (several blocks a head: 40 and 64 tokens), as many parts as there may be
@pytest.mark.parametrize("tokens,start,heads,kv,hd", [
    (1, 4000, 32, 8, 128), (1, 16001, 32, 8, 128), (5, 2047, 32, 8, 128), (16, 16368, 32, 8, 128), (40, 4090, 32, 8, 128),
    (64, 8000, 32, 8, 128), (130, 3967, 32, 8, 128), (1, 2112, 4, 2, 64), (33, 6001, 4, 2, 64), (3, 20000, 3, 1, 128),
    (2, 66000, 2, 1, 64)])
def test_attention_rows_behind_a_long_cache(tokens, start, heads, kv, hd):
    """The parts' fp32 shares are added up in fp32: the bound of the one-pass form.  The same call without a scratch
    (hqq_attention_rows) walks the positions in one block and gives the same within that bound."""
    from mixtral_offloading_amd import _lib, hip_kernels
    assert _parts(tokens, start, heads, kv, hd) > 1
    q, ck, cv = _case(tokens, start, heads, kv, hd, seed=tokens + start, spread=1.5)
    want, bound = _reference(q, ck, cv, start)
    for _ in range(2):
        got = hip_kernels.attention_rows(q, ck, cv, start).double().cpu()
        assert ((got - want).abs() <= 2 * bound).all()
    one = torch.empty((tokens, heads * hd), dtype=torch.float16, device="cuda")
    _lib.check(_lib.lib.hqq_attention_rows(q.data_ptr(), ck.data_ptr(), cv.data_ptr(), start, tokens, ck.shape[1], heads, kv, hd,
                                           one.data_ptr(), _lib.current_stream_ptr(q.device)), "hqq_attention_rows")
    assert ((one.double().cpu() - want).abs() <= 2 * bound).all()


@pytest.mark.parametrize("tokens,start", [(70, 100), (20, 5000)])  # one part; several
def test_attention_rows_infinities_and_nan_in_visible_positions(tokens, start):
    """What softmax gives in 64 bits: a key that is NaN or scores +inf makes the rows that see it NaN and leaves the
    others alone, one that scores -inf has no weight; an infinite or NaN value reaches its column of the rows that see it."""
    from mixtral_offloading_amd import hip_kernels
    heads, kv, hd = 8, 2, 128
    assert (_parts(tokens, start, heads, kv, hd) > 1) == (start == 5000)
    clean = _case(tokens, start, heads, kv, hd, seed=3)
    at = start + tokens // 2  # the second half of the tokens see it
    for value in (float("nan"), float("inf"), float("-inf")):
        q, ck, cv = (t.clone() for t in clean)
        ck[0, at, 5] = value
        want, bound = _reference(q, ck, cv, start)
        got = hip_kernels.attention_rows(q, ck, cv, start).double().cpu()
        assert torch.equal(got.isnan(), want.isnan()) and bool(want.isnan().any()) and bool((~want.isnan()[tokens // 2:]).any())
        seen = ~want.isnan()
        assert ((got - want).abs() <= 2 * bound)[seen].all()
        q, ck, cv = (t.clone() for t in clean)
        cv[0, 7, 5] = value  # every row sees it
        want, _ = _reference(q, ck, cv, start)
        got = hip_kernels.attention_rows(q, ck, cv, start).double().cpu()
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        assert torch.equal(got[got.isinf()], want[want.isinf()]) and bool((got.isinf() | got.isnan()).any())


def test_attention_rows_refuses_what_it_does_not_take():
    from mixtral_offloading_amd import hip_kernels
    q, ck, cv = _case(4, 0, 4, 2, 64)
    assert not hip_kernels.attention_rows_supported(q[..., :32].contiguous(), ck, cv)
    assert not hip_kernels.attention_rows_supported(q.transpose(0, 1), ck, cv)
    assert not hip_kernels.attention_rows_supported(q.float(), ck, cv)
    with pytest.raises(AssertionError):
        hip_kernels.attention_rows(q, ck, cv, 5)  # past the cache
