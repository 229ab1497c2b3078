"""Row copies: one launch for several, at every word size and over strided views, equal to torch's copies."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("shift", [0, 2, 1])  # elements the destination is off a 16-byte boundary by: words of 16, 4 and 2 bytes
@pytest.mark.parametrize("rows", [0, 1, 15, 33, 1000])
def test_row_copies_equal_torchs(rows: int, shift: int, dtype: torch.dtype) -> None:
    from lazykv_amd import kernels

    h, d = 3, 64
    gen = torch.Generator(device="cuda").manual_seed(rows)
    a = torch.randn((h, rows + 2, d), device="cuda", generator=gen).to(dtype)
    b = torch.randn((rows, h, d), device="cuda", generator=gen).to(dtype).transpose(0, 1)  # rows h * d apart
    flat = torch.zeros((2, h * (rows + 5) * d + 8), device="cuda", dtype=dtype)
    got = [f[shift : shift + h * (rows + 5) * d].view(h, rows + 5, d) for f in flat]
    kernels.copy_rows([(got[0][:, 3 : 3 + rows], a[:, 1 : 1 + rows]), (got[1][:, :rows], b), (got[1][:, rows : rows + 1], a[:, :1])])
    want = torch.zeros_like(flat)
    w = [f[shift : shift + h * (rows + 5) * d].view(h, rows + 5, d) for f in want]
    w[0][:, 3 : 3 + rows].copy_(a[:, 1 : 1 + rows])
    w[1][:, :rows].copy_(b)
    w[1][:, rows : rows + 1].copy_(a[:, :1])
    assert torch.equal(flat, want)


def test_copies_the_launch_does_not_cover_are_torchs() -> None:
    from lazykv_amd import kernels

    dst = torch.zeros((2, 4, 64), device="cuda", dtype=torch.bfloat16)
    src = torch.randn((2, 2, 64), device="cuda")
    kernels.copy_rows([(dst[:, :2], src), (dst[:, 2:3], src[:1, :1]), (dst[:, 3:], torch.ones((2, 1, 64)))])
    assert torch.equal(dst[:, :2], src.to(torch.bfloat16))
    assert torch.equal(dst[:, 2:3], src[:1, :1].to(torch.bfloat16).expand(2, 1, 64))
    assert torch.equal(dst[:, 3:], torch.ones((2, 1, 64), device="cuda", dtype=torch.bfloat16))
