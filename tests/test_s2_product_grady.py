"""The kernel gradient of the product on the sphere in the real basis: slices of every width, full and ragged tiles and passes."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [
    # one lane to sixty-four per slice and one more; loads of four, two and one
    (3, 1, 1, 4), (5, 7, 8, 4), (7, 3, 9, 1), (6, 40, 6, 20), (9, 5, 6, 100), (8, 2, 3, 256), (8, 3, 2, 260), (5, 4, 7, 26), (6, 3, 8, 63), (4, 6, 17, 65),
    # fewer pairs than slices, whole chunks of 256 pairs and one more, few and many workgroups
    (1, 1, 6, 8), (1, 256, 6, 8), (1, 257, 6, 8), (16, 32, 6, 100), (32, 9, 6, 100), (16, 20, 3, 45)])
def test_kernel_gradient(hip, nl, B, Fi, Fo):
    from s2cnn_amd.s2_real import s2_mm_real
    print(f"s2 kernel gradient nl={nl} B={B} Fi={Fi} Fo={Fo}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(nl)
    x = torch.randn(nl * nl, B, Fi, device="cuda", generator=g)
    y = torch.randn(nl * nl, Fi, Fo, device="cuda", generator=g).requires_grad_()
    z = s2_mm_real(x, y)
    gz = torch.randn(z.shape, device="cuda", generator=g)
    (gy,) = torch.autograd.grad(z, y, gz)
    for l in range(nl):
        L, first = 2 * l + 1, l * (4 * l * l - 1) // 3
        want = torch.einsum("rsij,rik->skj", gz[first:first + L * L].view(L, L, B, Fo).double(), x[l * l:l * l + L].double())
        got = gy[l * l:l * l + L].double()
        # sums of L B products, at most one rounding of 2^-24 each on partial sums that grow with the root of their number
        assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -24 * (1 + (L * B) ** 0.5)
