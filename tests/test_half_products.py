"""The forward products of long contractions, operand values cut into two f16 parts with a scale per row: at the edges of their tiles and
walks, and on values that the parts of a row do not represent together."""
import pytest
import torch

from oracle import cpu_path as O
from test_split_products import bound, product64, unaligned

# bound(K): six roundings per 16 steps.  Here there are three, and 2^-26.6 for the products of low parts that are left out.


def products(x, y, gz):
    import s2cnn_amd
    xg, yg = x.detach().requires_grad_(), y.detach().requires_grad_()
    z = s2cnn_amd.so3_mm_real(xg, yg)
    return (z.detach(), *torch.autograd.grad(z, (xg, yg), gz))


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [
    # blocks that the stage of 32 steps divides, that divide it (16, 8); granules of four steps; ragged tiles and last stages
    (16, 32, 64, 64), (25, 16, 16, 40), (49, 8, 8, 16), (16, 36, 60, 52), (16, 33, 28, 68), (17, 31, 100, 64),
    # beside them, what the rule leaves to the kernel of bf16 parts: short, odd, not aligned
    (16, 33, 24, 64), (16, 34, 50, 62)])
@pytest.mark.parametrize("aligned", [True, False])
def test_half_product_edges(hip, nl, B, Fi, Fo, aligned):
    print(f"half product nl={nl} B={B} Fi={Fi} Fo={Fo} aligned={aligned}", flush=True)
    ns = O.nspec_so3(nl)
    g = torch.Generator(device="cuda").manual_seed(nl)
    x, y, gz = (torch.randn(ns, *s, device="cuda", generator=g) for s in ((B, Fi), (Fi, Fo), (B, Fo)))
    if not aligned:
        x, y, gz = unaligned(x), unaligned(y), unaligned(gz)
    z, gx, gy = products(x, y, gz)
    L = 2 * nl - 1
    for got, want, K in ((z, product64("fwd", x, y, nl), L * Fi), (gx, product64("gradx", gz, y, nl), L * Fo), (gy, product64("grady", gz, x, nl), L * B)):
        assert ((got.double() - want).norm() / want.norm()).item() <= bound(K)


def rowwise(got, want, dim):
    """Largest relative error of the results of one index of `dim`; where the result is zero the difference has to be."""
    got, want = (t.movedim(dim, 0).flatten(1) for t in (got.double(), want))
    err, size = (got - want).norm(dim=1), want.norm(dim=1)
    assert torch.equal(err[size == 0], size[size == 0])
    return (err[size > 0] / size[size > 0]).max().item()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["zeros", "rows", "partners", "outlier", "channel", "tiny", "huge"])
def test_half_product_of_unequal_values(hip, kind):
    """Every row and column of the results as exact as float32 products are, whatever the sizes of the others: zeros, rows and columns of
    sizes of their own, large values beside small partners, a value that no sample shows, a row that meets small partners only."""
    nl, B, Fi, Fo = 16, 32, 60, 64
    ns, L = O.nspec_so3(nl), 2 * nl - 1
    print(f"half product of {kind}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    x, y, gz = (torch.randn(ns, *s, device="cuda", generator=g) for s in ((B, Fi), (Fi, Fo), (B, Fo)))
    sizes = lambda n, e: torch.exp2(torch.linspace(-e, e, n, device="cuda").round())  # noqa: E731
    if kind == "zeros":
        x[:, 3], x[:, :, 7], y[:, :, 5], y[:, 11] = 0.0, 0.0, 0.0, 0.0
    elif kind == "rows":
        x, y, gz = x * sizes(B, 50)[:, None], y * sizes(Fo, 50), gz * sizes(B, 20)[:, None]
    elif kind == "partners":
        x, y = x * sizes(Fi, 30), y * sizes(Fi, 30).flip(0)[:, None]
    elif kind == "outlier":
        x[ns - 100, 2, 9] = 2.0 ** 21
        y[ns - 77, 4, 6] = -(2.0 ** 23)
    elif kind == "channel":      # batch item 1 has one channel, which the kernel hardly takes
        x[:, 1, 1:] = 0.0
        y[:, 0] *= 2.0 ** -45
    elif kind == "tiny":
        x *= 2.0 ** -120
    else:
        x, y = x * 2.0 ** 60, y * 2.0 ** 50
    z, gx, gy = products(x, y, gz)
    assert rowwise(z, product64("fwd", x, y, nl), 1) <= 2 * bound(L * Fi) and rowwise(z, product64("fwd", x, y, nl), 2) <= 2 * bound(L * Fi)
    assert rowwise(gx, product64("gradx", gz, y, nl), 1) <= 2 * bound(L * Fo)
    if kind != "tiny":           # (results of subnormal size)
        assert rowwise(gy, product64("grady", gz, x, nl), 1) <= 2 * bound(L * B)


@pytest.mark.gpu
def test_half_product_of_values_that_are_not_finite(hip):
    nl, B, Fi, Fo = 16, 32, 60, 64
    ns = O.nspec_so3(nl)
    g = torch.Generator(device="cuda").manual_seed(5)
    x, y = torch.randn(ns, B, Fi, device="cuda", generator=g), torch.randn(ns, Fi, Fo, device="cuda", generator=g) * 0.125
    y[ns - 300:, :, 0] = 0.0
    plain = product64("fwd", x, y, nl)
    x[ns - 1, 0, 0] = float("inf")          # times zeros (NaN), times positive and negative values
    x[ns - 7, 1, 1] = float("nan")
    x[ns - 12, 2, 2] = 3.4e38 * 0.9999
    want = product64("fwd", x, y, nl)
    import s2cnn_amd
    got = s2cnn_amd.so3_mm_real(x, y).double()
    overflow = want.abs() > 3.402823466e38
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.isnan(want).any()
    assert torch.equal(got[overflow], want[overflow].sign() * float("inf"))
    ok = torch.isfinite(want) & ~overflow
    huge = ok & (want.abs() > 1e20)         # one huge product and terms that vanish beside it: two roundings
    assert huge.any() and ((got - want)[huge].abs() <= 2.0 ** -22 * want[huge].abs()).all()
    same = ok & ~huge
    assert ((got - plain)[same].norm() / want[same].norm()).item() <= bound((2 * nl - 1) * Fi)
