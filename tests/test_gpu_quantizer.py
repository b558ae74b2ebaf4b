"""The library's quantiser (hqq_quantize_groups / hqq_quantize_whole) against the oracle's restatement of hqq's
Quantizer.quantize.  Without the solver every output is a single correctly rounded fp32 operation of its inputs, so
codes, scale and zero must agree bit for bit; with the solver the shrinkage uses a power function whose last bit is
the library's own, so agreement is asked for up to a handful of codes on a rounding boundary.  (Both restate hqq from
memory: what is pinned here is that the GPU kernel and the CPU restatement are the same function, and, below, what the
mathematics fixes.)"""
import numpy as np
import pytest
import torch

from oracle import hqq_oracle as o

pytestmark = pytest.mark.gpu


def _weights(rng, n, k, dtype):
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    w[rng.integers(0, n, 8), rng.integers(0, k, 8)] *= 30.0  # a few outliers, as real weights have
    return w.astype(dtype)


@pytest.mark.parametrize("nbits,gs,round_zero", [(2, 16, False), (3, 64, False), (4, 64, True), (8, 128, False), (4, 32, False),
                                                 (2, 8, False)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_min_max_quantiser_equals_the_oracle_bit_for_bit(nbits, gs, round_zero, dtype):
    from mixtral_offloading_amd import hip_kernels
    rng = np.random.default_rng(nbits * 100 + gs)
    w = _weights(rng, 384, 320, dtype)
    q, scale, zero = o.hqq_quantize_tensor(w, nbits, gs, round_zero=round_zero)
    gq, gscale, gzero = hip_kernels.quantize_groups(torch.from_numpy(w).cuda(), gs, nbits, round_zero=round_zero)
    assert np.array_equal(gq.cpu().numpy(), q)
    assert np.array_equal(gscale.cpu().numpy().view(np.uint32), scale.reshape(1, -1).view(np.uint32))
    assert np.array_equal(gzero.cpu().numpy().view(np.uint32), zero.reshape(1, -1).view(np.uint32))


@pytest.mark.parametrize("gs,cols,off", [(16, 1613, 0), (32, 2047, 1), (64, 999, 2), (128, 2272, 3), (8, 1, 0), (16, 6, 1)])
def test_ragged_column_counts_and_unaligned_starts(gs, cols, off):
    """Column counts that are no multiple of the groups a thread takes, and tensors that start at any element of an
    allocation: the kernel falls back to narrower accesses and the result is the same."""
    from mixtral_offloading_amd import hip_kernels
    rng = np.random.default_rng(gs + cols)
    for dtype in (np.float16, np.float32):
        w = rng.standard_normal(gs * cols + off).astype(dtype)
        q, scale, zero = o.hqq_quantize_tensor(w[off:].reshape(gs, cols), 4, gs, round_zero=True)
        gq, gscale, gzero = hip_kernels.quantize_groups(torch.from_numpy(w).cuda()[off:], gs, 4, round_zero=True)
        assert np.array_equal(gq.cpu().numpy(), q)
        assert np.array_equal(gscale.cpu().numpy(), scale.reshape(1, -1)) and np.array_equal(gzero.cpu().numpy(), zero.reshape(1, -1))


def test_constant_and_tiny_groups():
    """max = min gives an infinite quotient that hqq clamps to 2e4; the codes are then all equal."""
    from mixtral_offloading_amd import hip_kernels
    w = np.zeros((64, 48), dtype=np.float32)
    w[:, 1] = 3.0
    w[:, 2] = np.linspace(0, 1e-6, 64)
    q, scale, zero = o.hqq_quantize_tensor(w, 4, 64)
    gq, gscale, gzero = hip_kernels.quantize_groups(torch.from_numpy(w).cuda(), 64, 4)
    assert np.array_equal(gq.cpu().numpy(), q)
    assert np.array_equal(gscale.cpu().numpy(), scale.reshape(1, -1)) and np.array_equal(gzero.cpu().numpy(), zero.reshape(1, -1))


@pytest.mark.parametrize("n", [1, 7, 4096, 100_003])
def test_whole_tensor_quantiser_equals_the_oracle(n):
    from mixtral_offloading_amd import hip_kernels
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n) * 3 + 1).astype(np.float32)
    q, scale, zero = o.hqq_quantize_tensor(x.reshape(1, n), 8, None, channel_wise=False)
    gq, gscale, gzero = hip_kernels.quantize_whole(torch.from_numpy(x).cuda().view(1, n), 8)
    assert np.array_equal(gq.cpu().numpy(), q.reshape(1, n))
    assert np.float32(gscale.item()) == np.float32(scale) and np.float32(gzero.item()) == np.float32(zero)


@pytest.mark.parametrize("nbits,gs", [(2, 16), (3, 64), (4, 64)])
def test_solver_agrees_with_the_oracle_and_lowers_the_error(nbits, gs):
    from mixtral_offloading_amd import hip_kernels
    rng = np.random.default_rng(7 + nbits)
    w = _weights(rng, 512, 256, np.float16)
    q, scale, zero = o.hqq_quantize_tensor(w, nbits, gs, optimize=True, round_zero=(nbits == 4))
    gq, gscale, gzero = hip_kernels.quantize_groups(torch.from_numpy(w).cuda(), gs, nbits, round_zero=(nbits == 4), iters=20)
    gq, gscale, gzero = gq.cpu().numpy(), gscale.cpu().numpy(), gzero.cpu().numpy()
    assert np.array_equal(gscale, scale.reshape(1, -1))  # the solver moves the zero only
    assert np.abs(gzero - zero.reshape(1, -1)).max() <= 1e-4 * (2 ** nbits)
    differ = gq != q
    assert differ.mean() <= 2e-4 and (not differ.any() or np.abs(gq.astype(int) - q.astype(int))[differ].max() == 1)
    # what the solver is for: a smaller l_p error (p = 0.7) of the reconstruction than plain min-max codes give
    wf = w.astype(np.float32).reshape(gs, -1)
    q0, s0, z0 = o.hqq_quantize_tensor(w, nbits, gs, round_zero=(nbits == 4))
    lp = lambda qq, ss, zz: float((np.abs(wf - (qq.astype(np.float32) - zz.reshape(1, -1)) * ss.reshape(1, -1)) ** 0.7).mean())  # noqa: E731
    assert lp(gq, gscale, gzero) < lp(q0, s0, z0)
    # and every code is the nearest level for the zero it ended with
    assert np.array_equal(gq, np.clip(np.round(wf / gscale + gzero), 0, 2 ** nbits - 1).astype(np.uint8)) or \
        (gq != np.clip(np.round(wf * (np.float32(1) / gscale) + gzero), 0, 2 ** nbits - 1)).mean() < 1e-3


def test_layer_quantised_on_the_gpu_equals_the_oracle_layer():
    """HQQLinearTritonSavable built from an fp16 nn.Linear on the GPU (codes through the quantiser, the packers and
    repack; 8-bit scale and zero tables through the quantiser again) against the oracle's layer, optimize off."""
    from mixtral_offloading_amd.custom_layers import HQQLinearTritonSavable
    from mixtral_offloading_amd.hqq_core import BaseQuantizeConfig
    rng = np.random.default_rng(3)
    for nbits, gs in [(2, 16), (3, 64), (4, 64)]:
        n, k = 640, 256
        w = _weights(rng, n, k, np.float16)
        cfg = BaseQuantizeConfig(nbits=nbits, group_size=gs, quant_zero=True, quant_scale=True)
        cfg["weight_quant_params"]["optimize"] = False
        lin = torch.nn.Linear(k, n, bias=False, dtype=torch.float16, device="cuda")
        lin.weight.data.copy_(torch.from_numpy(w))
        layer = HQQLinearTritonSavable(lin, cfg)
        want = o.hqq_quantize_layer(w, nbits, gs)
        assert np.array_equal(torch.Tensor.as_subclass(layer.W_q, torch.Tensor).cpu().numpy(), want["W_q"])
        assert np.array_equal(layer.meta["scale_q"].cpu().numpy(), want["scale_q"])
        assert np.array_equal(layer.meta["zero_q"].cpu().numpy().reshape(-1), want["zero_q"].reshape(-1))
        for t in ("meta_scale", "meta_zero"):
            for f in ("scale", "zero"):
                got = layer.meta[t][f].cpu().numpy().reshape(-1)
                assert np.array_equal(got.view(np.uint16), np.asarray(want[t][f], dtype=np.float16).reshape(-1).view(np.uint16)), (nbits, t, f)


@pytest.mark.parametrize("kind", ["wide", "constant", "huge", "offset"])
@pytest.mark.parametrize("nbits,gs", [(2, 8), (2, 16), (3, 64), (4, 128)])
def test_solver_where_its_short_cuts_do_not_hold(kind, nbits, gs):
    """Residuals large enough for the shrinkage to leave something (weights tens wide), groups without a spread, and
    scales and zeros outside the range in which a quotient is a product by the reciprocal in two floats: the tensor-op
    form's results.  The solver's zero is a mean of gs fp32 terms of size |w| * scale, so another order of that sum moves it by
    gs * 2^-24 of the largest."""
    from mixtral_offloading_amd import hip_kernels
    rng = np.random.default_rng(nbits * 1000 + gs)
    n, k = gs * 3, 84
    w = rng.standard_normal((n, k)).astype(np.float32)
    if kind == "wide":
        w *= 30
    elif kind == "constant":
        w[:, ::3] = 0.25
    elif kind == "huge":
        w[:, ::2] *= np.float32(2.0 ** 70)
    else:
        w = w * np.float32(1e-3) + 50
    q, scale, zero = o.hqq_quantize_tensor(w, nbits, gs, optimize=True, round_zero=(nbits == 4), iters=6)
    gq, gscale, gzero = hip_kernels.quantize_groups(torch.from_numpy(w).cuda(), gs, nbits, round_zero=(nbits == 4), iters=6)
    gq, gscale, gzero = gq.cpu().numpy(), gscale.cpu().numpy().reshape(-1), gzero.cpu().numpy().reshape(-1)
    assert np.array_equal(gscale, scale.reshape(-1))
    terms = np.abs(w.reshape(gs, -1).astype(np.float64) / scale.reshape(1, -1)).max(axis=0) + 2 ** nbits
    assert (np.abs(gzero - zero.reshape(-1)) <= 1e-4 * 2 ** nbits + 6 * gs * 2.0 ** -24 * terms).all()
    moved = np.abs(gq.astype(int) - q.astype(int))
    assert moved.max() <= 1 and (moved != 0).mean() <= (0.02 if kind == "offset" else 2e-3)


@pytest.mark.parametrize("nbits,gs,cols", [(2, 16, 4 * 256 * 1030 + 4), (3, 64, 2 * 256 * 70 + 2), (4, 64, 1), (2, 8, 256 * 1060 + 5)])
def test_solver_with_room_for_fewer_error_sums(nbits, gs, cols):
    """The solver's error is added up in as many places as the workspace holds and the blocks (1031, 71, 1 and 1061, one
    sum for 32 of them) are worth, down to one: the stop, and with it every output, is the same (the sums are fp64, and
    the stop compares their fp32 means).  The workspace starts as doubles of 1e306: a sum that is not cleared shows."""
    from mixtral_offloading_amd import _lib, hip_kernels
    gen = torch.Generator(device="cuda").manual_seed(cols)
    w = (torch.randn((gs, cols), device="cuda", generator=gen) * 0.02).half()
    want = hip_kernels.quantize_groups(w, gs, nbits, iters=20)
    full = int(_lib.lib.hqq_quantize_workspace_bytes())
    for nbytes in (64 * 8 + 64, 2 * 64 * 8 + 64, 7 * 64 * 8 + 100, full):
        ws = torch.full((nbytes + 64,), 0x7F, dtype=torch.uint8, device="cuda")
        got = [torch.empty_like(t) for t in want]
        rc = _lib.lib.hqq_quantize_groups(w.data_ptr(), 0, gs, cols, nbits, 0, 20, 0.7, 10.0, 1.01, got[0].data_ptr(),
                                          got[1].data_ptr(), got[2].data_ptr(), ws.data_ptr(), nbytes,
                                          _lib.current_stream_ptr(w.device))
        assert rc == 0
        assert all(torch.equal(a, b) for a, b in zip(got, want)), nbytes
        assert bool((ws[nbytes:] == 0x7F).all())  # nothing past the end it was told of
    assert _lib.lib.hqq_quantize_groups(w.data_ptr(), 0, gs, cols, nbits, 0, 20, 0.7, 10.0, 1.01, got[0].data_ptr(),
                                        got[1].data_ptr(), got[2].data_ptr(), ws.data_ptr(), 64 * 8 + 63,
                                        _lib.current_stream_ptr(w.device)) == -5


@pytest.mark.parametrize("gs,cols,sums", [(8, 1021, 1), (16, 4 * 256 * 63, 1), (16, 4 * 256 * 63 + 4, 2), (64, 2 * 256 * 96, 3)])
def test_tensors_of_few_blocks_use_few_error_sums(gs, cols, sums):
    """Every block of every pass reads all sums, so a tensor takes one for 32 of its blocks: the others are neither
    cleared nor added to."""
    from mixtral_offloading_amd import _lib, hip_kernels
    gen = torch.Generator(device="cuda").manual_seed(cols)
    w = (torch.randn((gs, cols), device="cuda", generator=gen) * 0.02).half()
    want = hip_kernels.quantize_groups(w, gs, 2, iters=20)
    got = [torch.empty_like(t) for t in want]
    ws = torch.full((int(_lib.lib.hqq_quantize_workspace_bytes()),), 0x7F, dtype=torch.uint8, device="cuda")
    assert _lib.lib.hqq_quantize_groups(w.data_ptr(), 0, gs, cols, 2, 0, 20, 0.7, 10.0, 1.01, got[0].data_ptr(),
                                        got[1].data_ptr(), got[2].data_ptr(), ws.data_ptr(), ws.numel(),
                                        _lib.current_stream_ptr(w.device)) == 0
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    err = ws[:sums * 512].view(torch.float64).view(sums, 64)
    assert bool((err[:, 0] > 0).all()) and bool((err < w.numel()).all())  # cleared, and each added to
    assert bool((ws[sums * 512:] == 0x7F).all())


@pytest.mark.parametrize("last", [5, 31])
def test_every_block_of_every_error_sum_counts_for_the_stop(last):
    """1061 blocks on 32 sums, so that most sums take a block of each of the 33 rounds.  The error lies in every 32nd
    block, all of one sum: with them the solver runs all 20 iterations, and what the other sums hold would stop it within
    10, which a fiftieth of the groups shows.  A rounding of the power or of a group's mean flips a code of a group now and
    then: a value has to lie within some 2^-21 of one of the three boundaries, in one of 8 x 20 looks, less than 1e-3 of
    the groups."""
    from mixtral_offloading_amd import _lib, hip_kernels
    gs, cols = 8, 256 * 1060 + 5  # odd: one group a thread
    rng = np.random.default_rng(last)
    w = rng.standard_normal((gs, cols)) * 0.02
    heavy = np.arange(cols) // 256 % 32 == last
    w[:, heavy] = rng.random((gs, int(heavy.sum()))) * 2
    w = w.astype(np.float16)
    q, scale, zero = o.hqq_quantize_tensor(w, 2, gs, optimize=True)
    # on the oracle: the other blocks alone stop within 10 iterations, and the tensor stopped there is another
    early = o.hqq_quantize_tensor(w[:, ~heavy], 2, gs, optimize=True, iters=10)[2]
    assert np.array_equal(early, o.hqq_quantize_tensor(w[:, ~heavy], 2, gs, optimize=True)[2])
    for iters in (10, 19):
        stopped = o.hqq_quantize_tensor(w, 2, gs, optimize=True, iters=iters)[2]
        assert (np.abs(stopped - zero) > 4e-4).mean() > 1e-2
    x = torch.from_numpy(w).cuda()
    gq, gscale, gzero = hip_kernels.quantize_groups(x, gs, 2, iters=20)
    assert np.array_equal(gscale.cpu().numpy(), scale.reshape(1, -1))
    assert (np.abs(gzero.cpu().numpy() - zero.reshape(1, -1)) > 4e-4).mean() <= 1e-3
    assert (gq.cpu().numpy() != q).mean() <= 1e-3
    # the first iteration's error, sum by sum, from the oracle's codes before it: block b in sum b % 32
    q0, s0, z0 = o.hqq_quantize_tensor(w, 2, gs)
    s0 = np.float32(1) / s0  # (the outputs hold 1 / scale; the error is made with scale, an ulp beside)
    err = np.abs(w.astype(np.float64) - (q0.astype(np.float64) - z0) / s0).sum(axis=0)
    want = np.bincount(np.arange(cols) // 256 % 32, weights=err, minlength=32)
    ws = torch.full((int(_lib.lib.hqq_quantize_workspace_bytes()),), 0x7F, dtype=torch.uint8, device="cuda")
    assert _lib.lib.hqq_quantize_groups(x.data_ptr(), 0, gs, cols, 2, 0, 20, 0.7, 10.0, 1.01, gq.data_ptr(), gscale.data_ptr(),
                                        gzero.data_ptr(), ws.data_ptr(), ws.numel(), _lib.current_stream_ptr(x.device)) == 0
    sums = ws[:32 * 512].view(torch.float64).view(32, 64)[:, 0].cpu().numpy()
    # a difference is good to some 2^-22 of its group's largest value, which is below ten times the mean difference, and
    # the roundings of 8 that are added may all go one way (a lost block would be a 33rd)
    assert np.allclose(sums, want, rtol=8 * 10 * 2.0 ** -22, atol=0)
