"""The end of a greedy decode step (reference: the sampling loop of transformers' ``generate`` with greedy settings):
logits copied, the first largest entry as the next token, the position one further.  Whole numbers: exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 9, 8191, 8192, 8200, 32000, 32768, 32771, 128257])
def test_next_token_is_torch_argmax(n):
    from mixtral_offloading_amd import hip_kernels
    gen = torch.Generator(device="cuda").manual_seed(n)
    base = torch.randn((1, n), device="cuda", generator=gen).half()
    rows = [base, -base.abs(), torch.zeros_like(base), base.round(), torch.full_like(base, float("-inf"))]
    for at in sorted({0, n // 2, n - 1}):  # one entry, in the first, a middle and the last place
        for value in (float("inf"), float("nan"), 100.0):
            row = base.clone()
            row[0, at] = value
            rows.append(row)
    signed = torch.zeros_like(base)
    signed[0, : n // 2] = -0.0
    rows.append(signed)
    pos = torch.full((1,), 5, dtype=torch.int64, device="cuda")
    for i, row in enumerate(rows):
        out, tok = torch.full_like(row, 3.0), torch.full((1,), -1, dtype=torch.int64, device="cuda")
        hip_kernels.next_token(row, out, tok, pos)
        host = row[0].cpu().float()
        nan = host.isnan()
        want = int(nan.nonzero()[0]) if bool(nan.any()) else int((host == host.max()).nonzero()[0])
        assert int(tok) == want and int(pos) == 6 + i
        assert torch.equal(out.view(torch.int16), row.view(torch.int16))


def test_next_token_refuses_misaligned_rows():
    from mixtral_offloading_amd import _lib, hip_kernels
    buf = torch.zeros(65, dtype=torch.float16, device="cuda")
    tok, pos = torch.zeros(1, dtype=torch.int64, device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    with pytest.raises(_lib.HqqError):
        hip_kernels.next_token(buf[1:], torch.zeros(64, dtype=torch.float16, device="cuda"), tok, pos)
