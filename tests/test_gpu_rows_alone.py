"""GPU parity tests of the rows kernel on one layer and on one expert (reference src/triton_kernels.py:137-212, a matmul over
quantised weights, and src/custom_layers.py:262-266) against de-quantise-then-matmul in fp32."""
import numpy as np
import pytest
import torch

from helpers import desc_of, launches
from oracle import hqq_oracle as o

pytestmark = pytest.mark.gpu

# (nbits, N, K, group size, 8-bit tables, rows): the edges of the 16-row tiles, of the cuts and of the rules' borders; K of four steps
# (one block along K) to 59 (several, the last one short); unit counts that do not fill the eight dies
CASES = [
    (2, 512, 512, 16, True, (17, 33, 64, 65)), (2, 1024, 3584, 16, True, (17, 32, 33, 129, 257, 640)),
    (2, 1152, 7552, 16, True, (31, 48, 97, 333)), (2, 768, 1152, 32, False, (40, 128, 200)),
    (4, 512, 512, 64, True, (33, 63, 64, 513)), (4, 1024, 3584, 64, True, (49, 96, 97, 193)),
    (4, 4224, 4096, 64, True, (17, 32, 288)), (4, 1152, 7552, 32, False, (65, 128, 333)),
    (3, 8192, 1536, 64, True, (17, 48, 64, 193)), (3, 3584, 8320, 64, True, (65, 100, 129)), (3, 3712, 1408, 128, False, (257, 319)),
]


def _close(got, x, d, bias=None):
    from mixtral_offloading_amd import hip_kernels
    w = hip_kernels.dequantize(d).float()
    ref = x.float() @ w.t()
    if bias is not None:
        ref = ref + bias.float()
    # fp16 weights rounded at other places and fp16 results: 1e-3 |x| |w| and a relative 1e-2, as for the other kernels
    bound = 1e-2 * ref.abs() + 1e-3 * x.float().norm(dim=1)[:, None] * w.norm(dim=1)[None, :]
    err = (got.float() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("case", CASES, ids=lambda c: "w%d_%dx%d_g%d_%s" % (*c[:4], "q" if c[4] else "f16"))
def test_one_layer_against_dequantize_then_matmul(case):
    from mixtral_offloading_amd import _lib, hip_kernels
    nbits, n, k, gs, tables, rows = case
    rng = np.random.default_rng(n + k + nbits)
    layer, _ = o.random_layer(rng, n, k, nbits, gs, tables, tables)
    bias = torch.from_numpy(rng.standard_normal(n).astype(np.float16)).cuda()
    d, db = desc_of(layer), desc_of(layer, bias=bias.cpu().numpy())
    gen = torch.Generator(device="cuda").manual_seed(n)
    for m in rows:
        x = torch.randn((m, k), device="cuda", generator=gen).half()
        got = hip_kernels.matmul(d, x)
        _close(got, x, d)
        assert torch.equal(got, hip_kernels.matmul(d, x))
        _close(hip_kernels.matmul(db, x), x, d, bias=bias)
        if hip_kernels.kernel_family(d, m) == _lib.FAM_TILE:
            # not the tile kernel's bits: the kernel under test has run (and at most one finishing pass)
            assert not torch.equal(got, hip_kernels.matmul(d, x, family=_lib.FAM_TILE))
            assert launches(lambda: hip_kernels.matmul(d, x)) <= 2


def test_rows_that_are_not_aligned_are_refused():
    from mixtral_offloading_amd import _lib, hip_kernels
    layer, _ = o.random_layer(np.random.default_rng(3), 512, 512, 2, 16)
    with pytest.raises(_lib.HqqError):
        hip_kernels.matmul(desc_of(layer), torch.zeros(64 * 512 + 1, device="cuda").half()[1:].view(64, 512))


@pytest.mark.parametrize("nbits,hidden,ffn,gs,rows", [
    (2, 1024, 3584, 16, (32, 33, 64, 65, 160, 300)), (2, 512, 7552, 16, (48, 129)), (4, 1024, 3584, 64, (17, 64, 97, 200)),
    (3, 1536, 3584, 64, (128, 129, 200, 400, 401))])
def test_one_expert_against_dequantize_then_matmul(nbits, hidden, ffn, gs, rows):
    from mixtral_offloading_amd import hip_kernels
    rng = np.random.default_rng(hidden + ffn + nbits)
    w1, w2, w3 = (desc_of(o.random_layer(rng, n, k, nbits, gs)[0]) for n, k in ((ffn, hidden), (hidden, ffn), (ffn, hidden)))
    wa, wc, wb = (hip_kernels.dequantize(d).float() for d in (w1, w2, w3))
    gen = torch.Generator(device="cuda").manual_seed(ffn)
    for m in rows:
        x = torch.randn((m, hidden), device="cuda", generator=gen).half()
        scale = (torch.rand((m,), device="cuda", generator=gen) * 0.6 + 0.2).half()
        h = torch.nn.functional.silu((x.float() @ wa.t()).half()) * (x.float() @ wb.t()).half()
        ref = h.float() @ wc.t()
        # four times the bound of one projection: h carries the tolerance of two already
        bound = 2e-2 * ref.abs() + 4e-3 * h.float().norm(dim=1)[:, None] * wc.norm(dim=1)[None, :]
        base = torch.randn((m, hidden), device="cuda", generator=gen).half()
        plain = hip_kernels.expert_ffn(w1, w2, w3, x)
        added = hip_kernels.expert_ffn(w1, w2, w3, x, out=base.clone(), row_scale=scale, accumulate=True)
        assert bool(((plain.float() - ref).abs() <= bound).all()), (m, float(((plain.float() - ref).abs() / bound).max()))
        err = (added.float() - (base.float() + ref * scale.float()[:, None])).abs()
        assert bool((err <= bound + 2e-3 * base.abs().float()).all()), (m, float((err / bound).max()))
