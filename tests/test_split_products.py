"""The block products on the bf16 matrix cores, every operand value cut into three bf16 parts: at the edges of their tiles and
walks over the contraction, on operands that are not aligned, and on values that the parts do not represent."""
import pytest
import torch

from oracle import cpu_path as O


def product64(which, a, b, nl):
    """The product of one degree after the other in float64: fwd (x, y), gradx (gz, y), grady (gz, x)."""
    out, pos = [], 0
    for l in range(nl):
        L = 2 * l + 1
        A = a[pos:pos + L * L].double().reshape(L, L, *a.shape[1:]).transpose(1, 2).reshape(L * a.shape[1], -1)      # (row, feature) x (col, feature)
        B = b[pos:pos + L * L].double().reshape(L, L, *b.shape[1:])
        if which == "grady":
            B = B.transpose(1, 2).reshape(L * b.shape[1], -1)
            Z = (A.t() @ B).reshape(L, a.shape[2], L, b.shape[2]).permute(0, 2, 3, 1)              # (n, j) x (p, k) as n, p, k, j
        else:
            B = B.permute(0, 3, 1, 2).reshape(L * b.shape[2], -1)                                  # (n, j) x (p, k)
            Z = (A @ (B.t() if which == "fwd" else B)).reshape(L, a.shape[1], L, -1).transpose(1, 2)
        out.append(Z.reshape(L * L, Z.shape[2], Z.shape[3]))
        pos += L * L
    return torch.cat(out)


def unaligned(t):
    """The same values behind a base that is aligned to 4 bytes only."""
    buf = torch.empty(t.numel() + 1, device=t.device)
    view = buf[1:].view(t.shape)
    return view.copy_(t)


# Errors: six roundings of 2^-24 per 16 contraction steps, of partial sums that grow with the root of the steps: about
# 2^-24 sqrt(6 K / 32 / 3) of the result, and one rounding for short contractions.  Twice that is allowed, and one more
# rounding: 2^-24 (1 + sqrt(K / 4)).
def bound(K):
    return 2.0 ** -24 * (1 + (K / 4) ** 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [
    # small problems, 32 x 32 and 32 x 64 outputs: one row, one block and one more, one 16-step and one more
    (1, 1, 1, 1), (1, 32, 16, 32), (1, 33, 17, 65), (3, 1, 7, 20), (6, 1, 20, 40), (7, 32, 100, 55), (2, 64, 65, 33),
    # tiles of 128 x 64 and 128 x 128, contraction blocks that divide the stage (8, 16, 32) or are divided by it (64)
    (16, 8, 40, 40), (12, 16, 64, 64), (10, 32, 96, 80),
    # granules of 4, 2 and 1 steps, ragged rows, columns and last stages, in the tiles of both widths
    (22, 3, 36, 20), (13, 11, 33, 45), (16, 9, 50, 70), (14, 13, 55, 41), (20, 7, 25, 60), (18, 30, 26, 38)])
@pytest.mark.parametrize("aligned", [True, False])
def test_real_product_edges(hip, nl, B, Fi, Fo, aligned):
    import s2cnn_amd
    print(f"split product nl={nl} B={B} Fi={Fi} Fo={Fo} aligned={aligned}", flush=True)
    ns = O.nspec_so3(nl)
    g = torch.Generator(device="cuda").manual_seed(nl)
    x, y, gz = (torch.randn(ns, *s, device="cuda", generator=g) for s in ((B, Fi), (Fi, Fo), (B, Fo)))
    if not aligned:
        x, y, gz = unaligned(x), unaligned(y), unaligned(gz)
    xg, yg = x.detach().requires_grad_(), y.detach().requires_grad_()
    z = s2cnn_amd.so3_mm_real(xg, yg)
    gx, gy = torch.autograd.grad(z, (xg, yg), gz)
    L = 2 * nl - 1
    for got, want, K in ((z, product64("fwd", x, y, nl), L * Fi), (gx, product64("gradx", gz, y, nl), L * Fo), (gy, product64("grady", gz, x, nl), L * B)):
        assert ((got.double() - want).norm() / want.norm()).item() <= bound(K)


def product64_complex(which, a, b, nl):
    """The same of complex operands [..., 2]: x conj(y), gz y, x conj(gz)."""
    (ar, ai), (br, bi) = a.unbind(-1), b.unbind(-1)
    ai, bi = -ai if which == "grady" else ai, -bi if which == "fwd" else bi
    return torch.stack((product64(which, ar, br, nl) - product64(which, ai, bi, nl),
                        product64(which, ai, br, nl) + product64(which, ar, bi, nl)), -1)


# The three real products of the Gauss form carry sqrt(2) times the error of a real product of the same length relative to the
# complex result (variances K + K of the real part, 4 K + K + K of the imaginary one, over 4 K), the sums of operands one more rounding.
@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [
    # 32 x 32 outputs: one row, one block and one more, one 16-step and one more
    (1, 1, 1, 1), (1, 32, 16, 32), (1, 33, 17, 65), (3, 1, 7, 20), (6, 1, 20, 40), (7, 32, 100, 55), (2, 64, 65, 33),
    # tiles of 128 x 128, contraction blocks that divide the stage (8, 16) or are divided by it (64), that neither
    (16, 8, 40, 40), (12, 16, 64, 64), (10, 32, 96, 80),
    # granules of 4, 2 and 1 steps, ragged rows, columns and last stages
    (22, 3, 36, 20), (16, 9, 50, 70), (14, 13, 55, 41), (20, 7, 25, 60), (18, 30, 26, 38)])
@pytest.mark.parametrize("aligned", [True, False])
def test_complex_product_edges(hip, nl, B, Fi, Fo, aligned):
    import s2cnn_amd
    print(f"complex split product nl={nl} B={B} Fi={Fi} Fo={Fo} aligned={aligned}", flush=True)
    ns = O.nspec_so3(nl)
    g = torch.Generator(device="cuda").manual_seed(nl)
    x, y, gz = (torch.randn(ns, *s, 2, device="cuda", generator=g) for s in ((B, Fi), (Fi, Fo), (B, Fo)))
    if not aligned:                       # to 8 bytes, the least that the library takes
        x, y, gz = (torch.empty(t.numel() + 2, device="cuda")[2:].view(t.shape).copy_(t) for t in (x, y, gz))
    xg, yg = x.detach().requires_grad_(), y.detach().requires_grad_()
    z = s2cnn_amd.so3_mm(xg, yg)
    gx, gy = torch.autograd.grad(z, (xg, yg), gz)
    L = 2 * nl - 1
    for got, want, K in ((z, product64_complex("fwd", x, y, nl), L * Fi), (gx, product64_complex("gradx", gz, y, nl), L * Fo),
                         (gy, product64_complex("grady", gz, x, nl), L * B)):
        assert ((got.double() - want).norm() / want.norm()).item() <= 2 * bound(K)


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [(3, 5, 9, 7), (16, 8, 40, 40)])      # either kernel
def test_complex_product_of_values_without_bf16_parts(hip, nl, B, Fi, Fo):
    """Results into which infinities, NaN or values that round to infinity in bf16 go are not finite where a float32 product is
    not, finite where it is, and the others are what they are without them."""
    import s2cnn_amd
    ns = O.nspec_so3(nl)
    g = torch.Generator(device="cuda").manual_seed(5)
    x, y = torch.randn(ns, B, Fi, 2, device="cuda", generator=g), torch.randn(ns, Fi, Fo, 2, device="cuda", generator=g) * 0.0625
    plain = product64_complex("fwd", x, y, nl)
    x[ns - 1, 0, 0, 0] = float("inf")
    x[ns - 7, 1, 1, 1] = float("nan")
    x[ns - 12, 2, 2, 0] = 3.4e38 * 0.9999   # its first bf16 part is infinite; its products are in range
    want = product64_complex("fwd", x, y, nl)
    got = s2cnn_amd.so3_mm(x, y).double()
    broken = ~torch.isfinite(want).all(-1)
    assert broken.any() and not torch.isfinite(got[broken]).all(-1).any()
    assert torch.isfinite(got[~broken]).all()
    # one huge product beside terms that vanish: three products of its size, rounded, and two sums of them: 2^-24 each, of a size
    # of up to |a||b| where the result may be a part of that
    huge = ~broken & (want.abs() > 1e20).any(-1)
    assert huge.any()
    size = want[huge].norm(dim=-1, keepdim=True)
    assert ((got - want)[huge].abs() <= 2.0 ** -21 * size).all()
    same = ~broken & ~huge
    assert ((got - plain)[same].norm() / want[same].norm()).item() <= 2 * bound((2 * nl - 1) * Fi)


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [(3, 5, 9, 7), (16, 8, 40, 40)])      # either kernel
def test_real_product_of_values_without_bf16_parts(hip, nl, B, Fi, Fo):
    """Infinities, NaN and values that round to infinity in bf16 give what float32 products give: where they take part
    the result is the infinity, NaN or finite value of the exact sum, and elsewhere nothing changes."""
    import s2cnn_amd
    ns = O.nspec_so3(nl)
    g = torch.Generator(device="cuda").manual_seed(5)
    x, y = torch.randn(ns, B, Fi, device="cuda", generator=g), torch.randn(ns, Fi, Fo, device="cuda", generator=g)
    y[ns - 30:, :, 0] = 0.0
    plain = product64("fwd", x, y, nl)
    x[ns - 1, 0, 0] = float("inf")          # times zeros (NaN), times positive and negative values
    x[ns - 7, 1, 1] = float("nan")
    x[ns - 12, 2, 2] = 3.4e38 * 0.9999      # its first bf16 part is infinite
    y = y * 0.125
    want = product64("fwd", x, y, nl)
    got = s2cnn_amd.so3_mm_real(x, y).double()
    assert (~torch.isfinite(want)).any() and torch.isfinite(want).any()
    overflow = want.abs() > 3.402823466e38
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[overflow], want[overflow].sign() * float("inf"))
    ok = torch.isfinite(want) & ~overflow
    # one huge product and terms that vanish beside it: the rounding of that product and of its sum, 2^-24 each
    huge = ok & (want.abs() > 1e20)
    assert huge.any() and ((got - want)[huge].abs() <= 2.0 ** -22 * want[huge].abs()).all()
    same = ok & ~huge
    assert ((got - plain * 0.125)[same].norm() / want[same].norm()).item() <= bound((2 * nl - 1) * Fi)


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [(3, 5, 9, 7), (16, 8, 40, 40)])      # either kernel
@pytest.mark.parametrize("complex_", [False, True])
def test_product_of_tiny_values(hip, nl, B, Fi, Fo, complex_):
    """Operands whose low bf16 parts are subnormal give the accuracy of float32 products: one rounding per step, twice what
    the sums of 16 steps are allowed."""
    import s2cnn_amd
    ns, pair = O.nspec_so3(nl), (2,) if complex_ else ()
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn(ns, B, Fi, *pair, device="cuda", generator=g) * 2.0 ** -118
    y = torch.randn(ns, Fi, Fo, *pair, device="cuda", generator=g)
    want = (product64_complex if complex_ else product64)("fwd", x, y, nl)
    got = (s2cnn_amd.so3_mm if complex_ else s2cnn_amd.so3_mm_real)(x, y)
    assert ((got.double() - want).norm() / want.norm()).item() <= 4 * bound((2 * nl - 1) * Fi)


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [(3, 5, 9, 7), (16, 8, 40, 40)])      # either kernel
@pytest.mark.parametrize("complex_", [False, True])
def test_product_of_tiny_values_and_large_partners(hip, nl, B, Fi, Fo, complex_):
    """The same where the other operand is large, so that the sums themselves are far from subnormal."""
    import s2cnn_amd
    ns, pair = O.nspec_so3(nl), (2,) if complex_ else ()
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn(ns, B, Fi, *pair, device="cuda", generator=g) * 2.0 ** -118
    y = torch.randn(ns, Fi, Fo, *pair, device="cuda", generator=g) * 2.0 ** 30
    want = (product64_complex if complex_ else product64)("fwd", x, y, nl)
    got = (s2cnn_amd.so3_mm if complex_ else s2cnn_amd.so3_mm_real)(x, y)
    assert ((got.double() - want).norm() / want.norm()).item() <= 4 * bound((2 * nl - 1) * Fi)


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [(3, 5, 9, 7), (16, 8, 40, 40)])      # either kernel
@pytest.mark.parametrize("complex_", [False, True])
@pytest.mark.parametrize("ex,ey", [(-118, 60), (-126, 60), (-140, 60), (-140, 100), (-60, -60), (30, 45), (105, -60)])
def test_products_over_the_exponents_of_float32(hip, nl, B, Fi, Fo, complex_, ex, ey):
    """Operands that are subnormal or next to it beside partners of any size, tiny products, scaled sums outside the range of float32:
    in both directions the errors of float32 products, one rounding per step."""
    import s2cnn_amd
    ns, pair = O.nspec_so3(nl), (2,) if complex_ else ()
    print(f"exponents nl={nl} B={B} Fi={Fi} Fo={Fo} complex={complex_} 2^{ex} 2^{ey}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(11)
    x, gz = ((torch.randn(ns, B, f, *pair, device="cuda", generator=g).double() * 2.0 ** ex).float() for f in (Fi, Fo))
    y = (torch.randn(ns, Fi, Fo, *pair, device="cuda", generator=g).double() * 2.0 ** ey).float()
    exact = product64_complex if complex_ else product64
    xg, yg = x.requires_grad_(), y.requires_grad_()
    z = (s2cnn_amd.so3_mm if complex_ else s2cnn_amd.so3_mm_real)(xg, yg)
    (gx,) = torch.autograd.grad(z, xg, gz)
    L = 2 * nl - 1
    for got, want, K in ((z.detach(), exact("fwd", x.detach(), y.detach(), nl), L * Fi), (gx, exact("gradx", gz, y.detach(), nl), L * Fo)):
        assert ((got.double() - want).norm() / want.norm()).item() <= 4 * bound(K)
    if ex < -100:      # grad y is a product of two operands of x's size: one of them as it is, the other of the size of y
        big = (torch.randn(ns, B, Fi, *pair, device="cuda", generator=g).double() * 2.0 ** ey).float().requires_grad_()
        zb = (s2cnn_amd.so3_mm if complex_ else s2cnn_amd.so3_mm_real)(big, yg)
        (gy,) = torch.autograd.grad(zb, yg, gz)
        want = exact("grady", gz, big.detach(), nl)
        assert ((gy.double() - want).norm() / want.norm()).item() <= 4 * bound(L * B)


# Operands beyond 32-bit byte offsets: 49 blocks of 2^24 floats at the top degree, 25 of complex numbers.  Loads of four, two
# and one, for x, y and gz the large operand.
@pytest.mark.gpu
@pytest.mark.parametrize("complex_,nl", [(False, 4), (True, 3)])
@pytest.mark.parametrize("B,Fi,Fo", [(3, 4096, 4096), (2, 4095, 4097), (2, 4094, 4098), (4096, 4096, 8), (4097, 4095, 3), (4096, 8, 4096), (4094, 6, 4097), (4094, 6, 4098)])
def test_products_of_operands_beyond_32_bit_offsets(hip, complex_, nl, B, Fi, Fo):
    import s2cnn_amd
    print(f"far product complex={complex_} nl={nl} B={B} Fi={Fi} Fo={Fo}", flush=True)
    ns, pair = O.nspec_so3(nl), (2,) if complex_ else ()
    g = torch.Generator(device="cuda").manual_seed(B)
    x, y, gz = (torch.randn(ns, *s, *pair, device="cuda", generator=g) for s in ((B, Fi), (Fi, Fo), (B, Fo)))
    z = (s2cnn_amd.so3_mm if complex_ else s2cnn_amd.so3_mm_real)(x.requires_grad_(), y.requires_grad_())
    gx, gy = torch.autograd.grad(z, (x, y), gz)
    l = nl - 1
    L, first = 2 * l + 1, O.nspec_so3(l)

    def matrix(t, columns_first):      # the top degree in float64, [(spectral row, feature row), (spectral column, feature column)] or transposed blocks
        t = t.detach()[first:].reshape(L, L, *t.shape[1:])
        t = torch.complex(t[..., 0].double(), t[..., 1].double()) if complex_ else t.double()
        return t.permute(1, 2, 0, 3).reshape(L * t.shape[2], -1) if columns_first else t.transpose(1, 2).reshape(L * t.shape[2], -1)

    def check(got, A, Bm, K):
        want = A @ Bm
        assert ((got - want).norm() / want.norm()).item() <= (2 if complex_ else 1) * bound(K)

    conj = (lambda t: t.conj()) if complex_ else (lambda t: t)
    X, Y, GZ = matrix(x, False), matrix(y, True), matrix(gz, False)      # Z = X Y^*, GX = GZ Y^T, GY: its blocks (column, row) X^T GZ^*
    check(matrix(z, False), X, conj(Y), L * Fi)
    check(matrix(gx, False), GZ, Y.t(), L * Fo)
    check(matrix(gy, True), X.t(), conj(GZ), L * B)


def chain(A, B, order):
    """A [M, K] B [K, N] in float32 as one chain of fused multiply-adds per entry (exact products; sums rounded to float64 on the way,
    which is another result once in 2^29 times)."""
    acc = torch.zeros(A.shape[0], B.shape[1], device=A.device)
    for k in order:
        acc = (A[:, k, None].double() * B[None, k].double() + acc.double()).float()
    return acc


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [(1, 1, 4, 1), (2, 3, 8, 5), (4, 33, 36, 7), (6, 32, 20, 40), (6, 1, 20, 40), (3, 70, 12, 33)])
def test_short_forward_products_are_chains(hip, nl, B, Fi, Fo):
    """Forward products of the small networks: every result is one chain in the order 8s + t, 8s + 4 + t, bit for bit.  A ReLU
    behind them takes a sample next to zero or leaves it by the last bit."""
    import s2cnn_amd
    ns = O.nspec_so3(nl)
    g = torch.Generator(device="cuda").manual_seed(nl)
    x, y = torch.randn(ns, B, Fi, device="cuda", generator=g), torch.randn(ns, Fi, Fo, device="cuda", generator=g)
    z = s2cnn_amd.so3_mm_real(x, y)
    pos = 0
    for l in range(nl):
        L = 2 * l + 1
        A = x[pos:pos + L * L].reshape(L, L, B, Fi).transpose(1, 2).reshape(L * B, L * Fi)
        Y = y[pos:pos + L * L].reshape(L, L, Fi, Fo).permute(1, 2, 0, 3).reshape(L * Fi, L * Fo)
        order = [8 * s + 4 * h + t for s in range((L * Fi + 7) // 8) for t in range(4) for h in range(2)]
        want = chain(A, Y, [k for k in order if k < L * Fi]).reshape(L, B, L, Fo).transpose(1, 2).reshape(L * L, B, Fo)
        assert torch.equal(z[pos:pos + L * L], want), l
        pos += L * L
