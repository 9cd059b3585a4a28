"""Kernel spectra of the layers (s2cnn_rft_planes, s2cnn_so3_rft and their adjoints) and the S^2 analysis that writes the real
basis, against float64 products with the matrices of the transforms."""
import numpy as np
import pytest
import torch

from oracle import cpu_path as O

pytestmark = pytest.mark.gpu


# Errors: products of K terms with six roundings of 2^-24 per 16 of them (about 2^-24 sqrt(K / 16) of the result), one rounding each
# of the matrix, the d-values and the factor, three of the sums over betas and the change of basis; all in relative 2-norm.
def bound(K):
    return 2.0 ** -24 * (6 + (K / 4) ** 0.5)


def rel(got, want):
    return ((got.double().cpu() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("b,shape", [
    (1, (1, 1)), (2, (1, 3)), (6, (20, 40)), (7, (3, 11)), (13, (33, 45)),          # split contraction, columns 1, 3, 800, 33, 1485
    (20, (32, 64)), (11, (5, 205))])                                             # a block per wave, whole and ragged columns
@pytest.mark.parametrize("kind", ["near", "equatorial", "point"])
def test_so3_kernel_spectrum(hip, b, shape, kind):
    import s2cnn_amd
    from s2cnn_amd import wigner
    from s2cnn_amd.so3_real import scaled_kernel_spectrum
    grid = {"near": s2cnn_amd.so3_near_identity_grid(), "equatorial": s2cnn_amd.so3_equatorial_grid(n_alpha=2 * b, n_beta=2, n_gamma=3),
            "point": ((0, 0, 0),)}[kind]
    print(f"kernel spectrum b={b} shape={shape} grid={kind}", flush=True)
    g = torch.Generator().manual_seed(b)
    k = torch.randn(*shape, len(grid), generator=g)
    F = torch.from_numpy(wigner.so3_ft_matrix_real(b, grid)) * 0.37
    kg = k.cuda().requires_grad_()
    y = scaled_kernel_spectrum(kg, 0.37, b, grid)
    gy = torch.randn(y.shape, generator=g)
    (gk,) = torch.autograd.grad(y, kg, gy.cuda())
    flat = k.double().reshape(-1, len(grid))
    assert rel(y.detach().reshape(F.size(1), -1), F.t() @ flat.t()) <= bound(len(grid))
    want = (gy.double().reshape(F.size(1), -1).t() @ F.t()).reshape(k.shape)
    # the sums over the spectrum cancel: the error is relative to |gy| |F|, as for any order of the sum
    size = ((gy.double().reshape(F.size(1), -1).t() ** 2) @ (F.t() ** 2)).sum().sqrt()
    assert ((gk.double().cpu() - want).norm() / size).item() <= bound(F.size(1))


@pytest.mark.parametrize("b,shape", [(1, (1, 1)), (10, (1, 20)), (20, (3, 26)), (32, (6, 100)), (7, (64, 320))])
def test_s2_kernel_spectrum(hip, b, shape):
    import s2cnn_amd
    from s2cnn_amd.s2_real import _setup_s2_ft_real, scaled_kernel_spectrum
    for grid in (s2cnn_amd.s2_near_identity_grid(), s2cnn_amd.s2_equatorial_grid(max_beta=0, n_alpha=130, n_beta=1)):
        g = torch.Generator().manual_seed(b)
        k = torch.randn(*shape, len(grid), generator=g)
        F = _setup_s2_ft_real(b, grid, torch.device("cpu")).double() * 0.37
        kg = k.cuda().requires_grad_()
        y = scaled_kernel_spectrum(kg, 0.37, b, grid)
        gy = torch.randn(y.shape, generator=g)
        (gk,) = torch.autograd.grad(y, kg, gy.cuda())
        assert rel(y.detach().reshape(F.size(1), -1), F.t() @ k.double().reshape(-1, len(grid)).t()) <= bound(len(grid))
        want = (gy.double().reshape(F.size(1), -1).t() @ F.t()).reshape(k.shape)
        size = ((gy.double().reshape(F.size(1), -1).t() ** 2) @ (F.t() ** 2)).sum().sqrt()
        assert ((gk.double().cpu() - want).norm() / size).item() <= bound(F.size(1))


def test_kernel_spectrum_of_values_without_bf16_parts(hip):
    """A column with an infinity or NaN is not finite; one with a value that rounds to infinity in bf16 and the others are."""
    import s2cnn_amd
    from s2cnn_amd import wigner
    from s2cnn_amd.so3_real import scaled_kernel_spectrum
    b, grid = 6, s2cnn_amd.so3_near_identity_grid()
    k = torch.randn(5, 9, len(grid), generator=torch.Generator().manual_seed(0))
    k[0, 0, 7], k[1, 1, 3], k[2, 2, 100] = float("inf"), float("nan"), 3.4e38 * 0.9999
    y = scaled_kernel_spectrum(k.cuda(), 0.0625, b, grid).cpu().reshape(-1, 45)
    finite = torch.isfinite(y).all(0)
    assert finite.sum() == 43 and not finite[0] and not finite[10]
    want = torch.from_numpy(wigner.so3_ft_matrix_real(b, grid)).t() @ k.double().reshape(45, -1)[finite].t() * 0.0625
    err = (y[:, finite].double() - want).norm(dim=0) / want.norm(dim=0)
    assert err.max().item() <= 4 * bound(len(grid))          # per column, with a quarter of the chip's columns as room


@pytest.mark.parametrize("ex", [-118, -128, -140])
def test_kernel_spectrum_gradients_of_tiny_values(hip, ex):
    """Incoming gradients that are subnormal or next to it, brought back by the factor: the accuracy of ordinary ones."""
    import s2cnn_amd
    from s2cnn_amd import wigner
    from s2cnn_amd.s2_real import _setup_s2_ft_real
    from s2cnn_amd import s2_real, so3_real
    b, scale = 10, 2.0 ** 100
    for mod, grid in ((so3_real, s2cnn_amd.so3_near_identity_grid()), (s2_real, s2cnn_amd.s2_near_identity_grid())):
        F = (torch.from_numpy(wigner.so3_ft_matrix_real(b, grid)) if mod is so3_real else _setup_s2_ft_real(b, grid, torch.device("cpu")).double()) * scale
        k = torch.randn(3, 20, len(grid), device="cuda").requires_grad_()
        y = mod.scaled_kernel_spectrum(k, scale, b, grid)
        gy = (torch.randn(y.shape, generator=torch.Generator().manual_seed(1)).double() * 2.0 ** ex).float()
        (gk,) = torch.autograd.grad(y, k, gy.cuda())
        flat = gy.double().reshape(F.size(1), -1).t()
        want = (flat @ F.t()).reshape(k.shape)
        # before the factor a gradient is rounded to float32, as a subnormal here: half of 2^-149.  So are the gradients of SO(3) plane
        # coefficients: b sums of a degree each and two of the change of basis, for each of the 2 b (2b - 1) coefficients that a sample's sum
        # takes, times up to 1
        slack = scale * 2.0 ** -150 * k.numel() ** 0.5 * (1 + ((b + 2) * 2 * b * (2 * b - 1) if mod is so3_real else 0))
        size = ((flat ** 2) @ (F.t() ** 2)).sum().sqrt()
        assert (gk.double().cpu() - want).norm().item() <= bound(F.size(1)) * size.item() + slack


def chain(A, B, order):
    """A [M, K] B [K, N] in float32 as one chain of fused multiply-adds per entry (exact products; sums rounded to float64 on the way,
    which is another result once in 2^29 times)."""
    acc = torch.zeros(A.shape[0], B.shape[1], device=A.device)
    for k in order:
        acc = (A[:, k, None].double() * B[None, k].double() + acc.double()).float()
    return acc


@pytest.mark.parametrize("b,shape", [(10, (1, 20)), (2, (1, 1)), (20, (3, 26))])
@pytest.mark.parametrize("n_alpha", [8, 5, 1])
def test_s2_kernel_spectra_of_small_layers_are_chains(hip, b, shape, n_alpha):
    """24, 15 and 3 points: one chain per entry, from the rounded product of kernel and factor, by 0 2 4 6 1 3 5 7 within each eight of the whole
    sixteens and the rest in sequence, bit for bit: what s2_rft_real's library product gave these layers (24 points)."""
    import s2cnn_amd
    from s2cnn_amd.s2_real import _setup_s2_ft_real, scaled_kernel_spectrum
    grid = s2cnn_amd.s2_near_identity_grid(n_alpha=n_alpha)
    P = len(grid)
    k = torch.randn(*shape, P, generator=torch.Generator().manual_seed(b)).cuda()
    m = P // 16 * 16
    order = [8 * s + t for s in range(m // 8) for t in (0, 2, 4, 6, 1, 3, 5, 7)] + list(range(m, P))
    F = _setup_s2_ft_real(b, grid, k.device)
    y = scaled_kernel_spectrum(k, 0.37, b, grid)
    assert torch.equal(y.reshape(F.size(1), -1), chain(F.t(), (k * 0.37).reshape(-1, P).t(), order))


@pytest.mark.parametrize("b,shape", [(6, (20, 40)), (2, (3, 4)), (5, (1, 36))])
def test_so3_kernel_spectra_of_small_layers_are_chains(hip, b, shape):
    """The plane coefficients of each beta as one chain over its points in their order, then the expansion: bit for bit the library product
    and expansion that these layers' spectra were formed with."""
    import s2cnn_amd
    from s2cnn_amd import _hip, wigner
    from s2cnn_amd.so3_real import scaled_kernel_spectrum
    grid = s2cnn_amd.so3_near_identity_grid()
    idx, E, dtab = wigner.so3_rft_plan(b, grid)
    E, dtab = (torch.from_numpy(t.astype(np.float32)).cuda().contiguous() for t in (E, dtab))
    k = torch.randn(*shape, len(grid), generator=torch.Generator().manual_seed(b)).cuda()
    ks = (k * 0.37).reshape(-1, len(grid))
    G = torch.stack([chain(E[i].t(), ks[:, torch.from_numpy(idx[i]).long().cuda()].t(), range(idx.shape[1])) for i in range(len(idx))]).contiguous()
    want = torch.empty(O.nspec_so3(b), ks.size(0), device="cuda")
    _hip.call("s2cnn_so3_rft_expand_real", _hip.ptr(G), _hip.ptr(dtab), _hip.ptr(want), b, len(idx), ks.size(0), _hip.stream_ptr())
    assert torch.equal(scaled_kernel_spectrum(k, 0.37, b, grid).reshape(want.shape), want)


@pytest.mark.parametrize("b,shape,points", [(13, (33, 45), 64), (20, (32, 40), 128), (7, (64, 320), 130)])
def test_tiled_kernel_spectrum_of_values_without_bf16_parts(hip, b, shape, points):
    """The same in tiles of 128 x 128: three betas of 64 points, one of 128, and a spectrum of the sphere."""
    import s2cnn_amd
    from s2cnn_amd import s2_real, so3_real, wigner
    n = shape[0] * shape[1]
    print(f"tiled kernel spectrum b={b} columns={n} points={points}", flush=True)
    if points == 130:
        mod, grid = s2_real, s2cnn_amd.s2_equatorial_grid(max_beta=0, n_alpha=130, n_beta=1)
        F = s2_real._setup_s2_ft_real(b, grid, torch.device("cpu")).double()
    else:
        mod = so3_real
        grid = s2cnn_amd.so3_near_identity_grid() if points == 64 else s2cnn_amd.so3_equatorial_grid(max_beta=0, max_gamma=0, n_alpha=128, n_beta=1, n_gamma=1)
        F = torch.from_numpy(wigner.so3_ft_matrix_real(b, grid))
    k = torch.randn(n, len(grid), generator=torch.Generator().manual_seed(0))
    k[0, 7], k[130, 3], k[257, 60], k[n - 1, 1] = float("inf"), float("nan"), 3.4e38 * 0.9999, 2.0 ** 105
    y = mod.scaled_kernel_spectrum(k.cuda().view(*shape, -1), 0.0625, b, grid).cpu().reshape(-1, n)
    finite = torch.isfinite(y).all(0)
    assert finite.sum() == n - 2 and not finite[0] and not finite[130]
    want = F.t() @ k.double()[finite].t() * 0.0625
    err = (y[:, finite].double() - want).norm(dim=0) / want.norm(dim=0)
    assert err.max().item() <= 4 * bound(len(grid))          # per column, with a quarter of the chip's columns as room


def test_kernel_spectrum_gradient_of_the_gradient(hip):
    """The transform is linear: the gradient of a function of its gradient is the transform again."""
    import s2cnn_amd
    from s2cnn_amd import s2_real, so3_real
    for mod, grid in ((so3_real, s2cnn_amd.so3_near_identity_grid()), (s2_real, s2cnn_amd.s2_near_identity_grid())):
        k = torch.randn(3, 5, len(grid), device="cuda", requires_grad=True)
        y = mod.scaled_kernel_spectrum(k, 0.5, 5, grid)
        gy = torch.randn_like(y).requires_grad_()
        (gk,) = torch.autograd.grad(y, k, gy, create_graph=True)
        v = torch.randn_like(gk)
        (ggy,) = torch.autograd.grad(gk, gy, v)
        assert torch.equal(ggy, mod.scaled_kernel_spectrum(v, 0.5, 5, grid))


@pytest.mark.parametrize("b_in,b_out,batch", [(1, 1, 1), (3, 2, 5), (30, 10, 1), (30, 10, 33), (50, 20, 27), (64, 32, 7), (128, 32, 3)])
def test_s2_analysis_in_the_real_basis(hip, b_in, b_out, batch):
    """The map of the complex spectrum and, as its gradient, that of the composition: the same sums in the same order, one more
    rounding of the factor."""
    from s2cnn_amd.s2_real import s2_spectrum_to_real
    from s2cnn_amd.soft.s2_fft import S2_fft_real, s2_rfft_real_basis
    x = torch.randn(batch, 1, 2 * b_in, 2 * b_in, device="cuda", requires_grad=True)
    want, got = s2_spectrum_to_real(S2_fft_real.apply(x, b_out)), s2_rfft_real_basis(x, b_out)
    assert got.shape == want.shape
    assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -22
    g = torch.randn_like(want)
    gw, gg = (torch.autograd.grad(y, x, g)[0] for y in (want, got))
    assert ((gg - gw).norm() / gw.norm()).item() <= 2.0 ** -22


@pytest.mark.parametrize("ncols", [4, 36, 1028])
def test_expansions_alone(hip, ncols):
    """The expansion over the degrees and its adjoint as entry points of their own, behind and in front of the products that s2cnn_so3_rft and its
    adjoint run: the same bits; the complex one against its change of basis."""
    import s2cnn_amd
    from s2cnn_amd import _hip, so3_real
    b, grid = 5, s2cnn_amd.so3_near_identity_grid()
    idx, E, Et, dtab = so3_real._setup_so3_rft_plan(b, grid, torch.device("cuda", torch.cuda.current_device()))
    (nbeta, P), R, npts, ns = idx.shape, E.size(2), len(grid), O.nspec_so3(b)
    P_, st = _hip.ptr, _hip.stream_ptr()
    g = torch.Generator(device="cuda").manual_seed(ncols)
    x, gy = torch.randn(ncols, npts, device="cuda", generator=g), torch.randn(ns, ncols, device="cuda", generator=g)
    G, gG = torch.empty(nbeta, R, ncols, device="cuda"), torch.empty(nbeta, R, ncols, device="cuda")
    y, yc, gx = torch.empty(ns, ncols, device="cuda"), torch.empty(ns, ncols, 2, device="cuda"), torch.empty(ncols, npts, device="cuda")
    _hip.call("s2cnn_rft_planes", P_(x), P_(idx), P_(E), P_(G), nbeta, P, R, npts, ncols, ncols, 0.5, st)
    _hip.call("s2cnn_so3_rft_expand_real", P_(G), P_(dtab), P_(y), b, nbeta, ncols, st)
    _hip.call("s2cnn_so3_rft_expand", P_(G), P_(dtab), P_(yc), b, nbeta, ncols, st)
    _hip.call("s2cnn_so3_rft_expand_real_grad", P_(gy), P_(dtab), P_(gG), b, nbeta, ncols, st)
    _hip.call("s2cnn_rft_planes_grad", P_(gG), P_(idx), P_(Et), P_(gx), nbeta, P, R, npts, ncols, ncols, 0.5, st)
    xg = x.clone().requires_grad_()
    want = so3_real._KernelSpectrum.apply(xg, b, (idx, E, Et, dtab), 0.5)
    (wgx,) = torch.autograd.grad(want, xg, gy)
    assert torch.equal(y, want) and torch.equal(gx, wgx)
    back = so3_real.so3_spectrum_to_real(yc)      # sums of two products with 1/sqrt2 or sqrt2: a few roundings
    assert ((back - y).norm() / y.norm()).item() <= 2.0 ** -22
