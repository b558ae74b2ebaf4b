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


@pytest.mark.parametrize("tokens,spread", [(2048, 1.0), (2100, 6.0)])
def test_attention_rows_two_tiles_a_wave(tokens, spread):
    """From 512 blocks a wave takes two query tiles (32 heads on 8 key/value heads: 2017 tokens)."""
    from mixtral_offloading_amd import hip_kernels
    q, ck, cv = _case(tokens, 5, 32, 8, 128, seed=tokens, spread=spread)
    want, bound = _reference(q, ck, cv, 5)
    got = hip_kernels.attention_rows(q, ck, cv, 5).double().cpu()
    assert ((got - want).abs() <= 2 * bound).all()


def test_attention_rows_refuses_what_it_does_not_take():
    from mixtral_offloading_amd import hip_kernels
    q, ck, cv = _case(4, 0, 4, 2, 64)
    assert not hip_kernels.attention_rows_supported(q[..., :32].contiguous(), ck, cv)
    assert not hip_kernels.attention_rows_supported(q.transpose(0, 1), ck, cv)
    assert not hip_kernels.attention_rows_supported(q.float(), ck, cv)
    with pytest.raises(AssertionError):
        hip_kernels.attention_rows(q, ck, cv, 5)  # past the cache
