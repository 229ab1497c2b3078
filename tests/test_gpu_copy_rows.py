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


def test_odd_bytes_are_torchs() -> None:
    from lazykv_amd import kernels

    src = torch.randint(0, 256, (3, 5, 7), dtype=torch.uint8, device="cuda")  # rows of 7 bytes
    dst = torch.zeros_like(src)
    even = torch.randint(0, 256, (3, 5, 9), dtype=torch.uint8, device="cuda")
    one_off = torch.zeros((3, 5, 9), dtype=torch.uint8, device="cuda")
    kernels.copy_rows([(dst, src), (one_off[:, :, 1:], even[:, :, 1:])])  # and rows of 8 at odd addresses
    assert torch.equal(dst, src) and torch.equal(one_off[:, :, 1:], even[:, :, 1:])
    src = torch.randn((70000, 1, 4), device="cuda")  # more heads than a launch has
    dst = torch.zeros_like(src)
    kernels.copy_rows([(dst, src)])
    assert torch.equal(dst, src)
    many = [(torch.zeros((2, 3, 64), device="cuda"), torch.randn((2, 3, 64), device="cuda")) for _ in range(19)]  # three launches
    kernels.copy_rows(many)
    assert all(torch.equal(d, s) for d, s in many)


def test_a_graph_that_saved_the_destination_sees_the_write() -> None:
    from lazykv_amd import kernels

    dst = torch.ones((2, 4, 64), device="cuda")
    w = torch.ones((2, 4, 64), device="cuda", requires_grad=True)
    y = (w * dst).sum()  # saves dst for w's gradient
    kernels.copy_rows([(dst[:, 1:3], torch.zeros((2, 2, 64), device="cuda"))])
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()


def test_tangents_are_copied() -> None:
    import torch.autograd.forward_ad as fw

    from lazykv_amd import kernels

    src, tangent = torch.randn((2, 3, 64), device="cuda"), torch.randn((2, 3, 64), device="cuda")
    with fw.dual_level():
        dst = torch.zeros((2, 4, 64), device="cuda")
        kernels.copy_rows([(dst[:, 1:], fw.make_dual(src, tangent))])
        got = fw.unpack_dual(dst)
        assert torch.equal(got.primal[:, 1:], src)
        assert got.tangent is not None and torch.equal(got.tangent[:, 1:], tangent)
        kernels.copy_rows([(dst[:, 1:], src)])  # a plain source clears them
        assert torch.equal(fw.unpack_dual(dst).tangent[:, 1:], torch.zeros_like(src))
