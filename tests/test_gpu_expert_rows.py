"""GPU parity tests of the experts of a MoE layer in common launches (``expert_rows_ffn``: reference
src/custom_layers.py:298-312 over rows grouped by expert) against de-quantise-then-matmul in fp32."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import desc_of, launches
from oracle import hqq_oracle as o

pytestmark = pytest.mark.gpu

# rows of the groups, at the edges of the 16-row tiles, of the two kernels (32 rows) and of a block's most tiles (96 and
# 128 rows), enough groups for the common launches
FEW = [1, 2, 15, 16, 17, 31, 32, 0, 3, 5, 8, 1, 30, 4, 18, 9, 2, 1, 16, 7, 11, 32]
MANY = [33, 48, 49, 64, 65, 80, 96, 97, 112, 113, 128, 129, 1, 16, 0, 200]
FEW3 = [1, 2, 15, 16, 17, 31, 32, 0] * 2 + [3, 5, 8, 1, 30, 4, 18, 9, 2, 1, 16, 7, 11, 32]  # (a block is four windows of 56)
# (nbits, hidden, ffn, group size, 8-bit tables, rows of the groups)
CASES = [
    (2, 1024, 3584, 16, True, FEW), (2, 1024, 3584, 16, True, MANY),
    (2, 512, 7552, 16, True, FEW), (2, 512, 7552, 16, True, MANY),  # down projections of 59 steps: two and more blocks along K
    (2, 1152, 3712, 16, True, FEW), (2, 1152, 3712, 16, True, MANY),  # 58 packed rows (a last block with rows to spare), 29 steps
    (2, 896, 3840, 32, False, FEW), (2, 896, 3840, 32, False, MANY),  # fp16 tables, two row blocks of a packed row
    (4, 1024, 3584, 64, True, FEW), (4, 1024, 3584, 64, True, MANY),
    (4, 1152, 3712, 32, False, MANY),
    # 3-bit: 28 windows of 13 word rows, the last of them with fields to spare (3584 rows are 358 words and four fields)
    (3, 1536, 3584, 64, True, FEW3), (3, 1536, 3584, 64, True, MANY),
    (3, 1536, 7552, 64, True, MANY),  # 59 windows (a block with some to spare), K split
    (3, 3456, 3712, 128, False, MANY),  # fp16 tables, 27 and 29 windows one table row apart
]


def _experts(nbits, hidden, ffn, gs, tables, count=3):
    rng = np.random.default_rng(hidden + ffn + nbits)
    shapes = ((ffn, hidden), (hidden, ffn), (ffn, hidden))
    bias = rng.standard_normal(hidden).astype(np.float16)  # of one expert's down projection
    layers = [[o.random_layer(rng, n, k, nbits, gs, tables, tables)[0] for n, k in shapes] for _ in range(count)]
    return [(desc_of(w1), desc_of(w2, bias=bias if i == 1 else None), desc_of(w3)) for i, (w1, w2, w3) in enumerate(layers)], bias


@pytest.mark.parametrize("case", CASES, ids=lambda c: "w%d_h%d_f%d_g%d_%s_%d" % (*c[:4], "q" if c[4] else "f16", len(c[5])))
def test_expert_rows_against_dequantize_then_matmul(case):
    from mixtral_offloading_amd import hip_kernels
    nbits, hidden, ffn, gs, tables, counts = case
    experts, bias = _experts(nbits, hidden, ffn, gs, tables)
    group = hip_kernels.ExpertGroup([experts[g % 3] for g in range(len(counts))])
    starts = np.concatenate(([0], np.cumsum(counts)))
    rows = int(starts[-1])
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn((rows, hidden), device="cuda", generator=gen).half()
    scale = (torch.rand((rows,), device="cuda", generator=gen) * 0.6 + 0.2).half()
    assert launches(lambda: hip_kernels.expert_rows_ffn(group, x, starts, scale, torch.empty_like(x))) <= 8
    outs = []
    for row_scale in (scale, None, scale):
        out = torch.full((rows, hidden), 7.0, dtype=torch.float16, device="cuda")
        hip_kernels.expert_rows_ffn(group, x, starts, row_scale, out)
        outs.append(out)
    assert torch.equal(outs[0], outs[2])
    weights = [[hip_kernels.dequantize(d).float() for d in e] for e in experts]
    for g, m in enumerate(counts):
        lo, hi = int(starts[g]), int(starts[g]) + m
        wa, wc, wb = weights[g % 3]
        a, b = (x[lo:hi].float() @ wa.t()).half(), (x[lo:hi].float() @ wb.t()).half()
        h = torch.nn.functional.silu(a) * b
        ref = h.float() @ wc.t() + (torch.from_numpy(bias).cuda().float() if g % 3 == 1 else 0.0)
        # four times the bound of one projection, 1e-3 |x| |w|: h carries the tolerance of two already
        bound = 2e-2 * ref.abs() + 4e-3 * h.float().norm(dim=1)[:, None] * wc.norm(dim=1)[None, :]
        for out, s in ((outs[0], scale[lo:hi, None].float()), (outs[1], 1.0)):
            err = (out[lo:hi].float() - ref * s).abs()
            assert bool((err <= bound).all()), (g, m, float((err / bound).max()))


@pytest.mark.parametrize("counts", [FEW, MANY, [1, 2, 5]])
def test_groups_that_are_left_out_change_nothing(counts):
    """The experts of a layer one at a time, as they arrive from host memory: each call writes its own rows, with the bits
    of all experts in one call.  A plan of few blocks is one hqq_expert_ffn per group."""
    from mixtral_offloading_amd import hip_kernels
    experts, _ = _experts(2, 1024, 3584, 16, True)
    every = [experts[g % 3] for g in range(len(counts))]
    starts = np.concatenate(([0], np.cumsum(counts)))
    rows = int(starts[-1])
    x = torch.randn((rows, 1024), device="cuda", generator=torch.Generator(device="cuda").manual_seed(rows)).half()
    want, got = torch.full_like(x, 3.0), torch.full_like(x, 5.0)
    hip_kernels.expert_rows_ffn(hip_kernels.ExpertGroup(every), x, starts, None, want)
    for g, m in enumerate(counts):
        if m:
            before = got.clone()
            hip_kernels.expert_rows_ffn(hip_kernels.ExpertGroup([e if i == g else None for i, e in enumerate(every)]), x, starts, None, got)
            keep = torch.ones(rows, dtype=torch.bool, device="cuda")
            keep[int(starts[g]):int(starts[g + 1])] = False
            assert torch.equal(got[keep], before[keep])
    assert torch.equal(got, want)
    if counts == [1, 2, 5]:
        hip_kernels.expert_groups_ffn(hip_kernels.ExpertGroup(every), x, starts, None, got)
        assert torch.equal(got, want)


def test_expert_rows_refuses_what_does_not_hold_it():
    from mixtral_offloading_amd import _lib, hip_kernels
    experts, _ = _experts(2, 1024, 3584, 16, True)
    group = hip_kernels.ExpertGroup([experts[g % 3] for g in range(len(FEW))])
    starts = (ctypes.c_int64 * (len(FEW) + 1))(*[int(v) for v in np.concatenate(([0], np.cumsum(FEW)))])
    rows = sum(FEW)
    x = torch.zeros((rows, 1024), dtype=torch.float16, device="cuda")
    need = _lib.lib.hqq_expert_rows_ffn_workspace_bytes(group.w1, group.w2, group.w3, group.n, starts)
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    args = (group.w1, group.w2, group.w3, group.n, starts, x.data_ptr(), x.data_ptr(), None, ws.data_ptr())
    stream = _lib.current_stream_ptr(x.device)
    assert _lib.lib.hqq_expert_rows_ffn(*args, need - 256, stream) == -5
    assert _lib.lib.hqq_expert_rows_ffn(*args[:5], None, *args[6:], need, stream) == -1
    starts[3] = 1
    assert _lib.lib.hqq_expert_rows_ffn(*args, need, stream) == -3
