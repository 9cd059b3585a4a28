"""The kernel gradient of the product on the sphere in the real basis: slices of every width, full and ragged tiles and passes."""
import ctypes
import os
import shutil
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    """The rule of the launch, compiled for the host: lanes(nl, f_in, groups of features in a row)."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    d = tmp_path_factory.mktemp("split")
    (d / "split.cpp").write_text('#include "s2_mm_real_tiles.h"\n'
                                 'extern "C" int lanes(int nl, int f_in, int fov) { return s2cnn::grady_lanes(nl, f_in, fov); }\n')
    subprocess.run([gxx, "-shared", "-fPIC", "-I", os.path.join(ROOT, "s2cnn_amd", "csrc"), str(d / "split.cpp"), "-o", str(d / "split.so")], check=True)
    return ctypes.CDLL(str(d / "split.so"))


def test_rows_are_cut_only_where_workgroups_are_few(split):
    for nl, Fi, fov, want in [(16, 6, 25, 13), (16, 25, 25, 25), (16, 32, 25, 25), (24, 32, 25, 25), (12, 64, 64, 64), (32, 6, 25, 25), (10, 1, 5, 5), (5, 8, 1, 4)]:
        assert split.lanes(nl, Fi, fov) == want, (nl, Fi, fov)
    for nl in range(1, 40):
        for Fi in (1, 8, 9, 16, 17, 64):
            passes = (Fi + 7) // 8
            for fov in range(1, 400):
                jt = split.lanes(nl, Fi, fov)
                tiles = -(-fov // jt)
                assert 4 <= jt <= 64
                if tiles > -(-fov // 64):                       # cut further: too few workgroups with half the tiles, and no slice under 9 lanes
                    assert nl * nl * passes * ((tiles + 1) // 2) < 1024 and jt >= 9


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
