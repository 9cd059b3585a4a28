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
    """The rule of the launch, compiled for the host: split(nl, batch, f_in, groups of features in a row) -> (lanes, slices)."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    d = tmp_path_factory.mktemp("split")
    (d / "split.cpp").write_text('#include "s2_mm_real_tiles.h"\n'
                                 'extern "C" int lanes(int nl, int b, int f, int v) { return s2cnn::grady_split(nl, b, f, v).lanes; }\n'
                                 'extern "C" int slices(int nl, int b, int f, int v) { return s2cnn::grady_split(nl, b, f, v).slices; }\n')
    subprocess.run([gxx, "-shared", "-fPIC", "-I", os.path.join(ROOT, "s2cnn_amd", "csrc"), str(d / "split.cpp"), "-o", str(d / "split.so")], check=True)
    lib = ctypes.CDLL(str(d / "split.so"))
    return lambda *size: (lib.lanes(*size), lib.slices(*size))


def test_rows_are_cut_only_where_workgroups_are_few(split):
    for nl, B, Fi, fov, want in [(16, 32, 6, 25, 13), (16, 32, 25, 25, 25), (16, 32, 32, 25, 25), (24, 16, 32, 25, 25), (12, 4, 64, 64, 64), (32, 32, 6, 25, 25),
                                 (10, 32, 1, 5, 5), (5, 7, 8, 1, 4),
                                 # few pairs for each slice
                                 (18, 2, 7, 37, 19), (9, 1, 20, 193, 49), (16, 1, 6, 25, 25), (22, 2, 4, 23, 23),
                                 # few pairs, but fewer workgroups than CUs
                                 (3, 7, 5, 56, 14), (5, 3, 60, 51, 26)]:
        assert split(nl, B, Fi, fov)[0] == want, (nl, B, Fi, fov)
    for nl in range(1, 40):
        for B in (1, 2, 9, 32, 1000):
            for Fi in (1, 8, 9, 64):
                passes, pairs = (Fi + 7) // 8, (2 * nl - 1) * B
                for fov in range(1, 300):
                    lanes, slices = split(nl, B, Fi, fov)
                    tiles = -(-fov // lanes)
                    assert 4 <= lanes <= 64 and 1 <= slices and lanes * slices <= 256
                    assert slices == min(256 // lanes, -(-pairs // 4))              # four pairs for each
                    if tiles > -(-fov // 64):             # cut further: too few workgroups with half the tiles, no slice under 9 lanes, five pairs or idle CUs
                        before = nl * nl * passes * ((tiles + 1) // 2)
                        assert before < 1024 and lanes >= 9 and (before < 256 or pairs // (256 // lanes) >= 5)


# (nl, B, Fi, Fo, elements by which gz starts beyond a boundary of 16 bytes)
SIZES = [
    # narrow slices, loads of four, two and one
    (3, 1, 1, 4, 0), (5, 7, 8, 4, 0), (7, 3, 9, 1, 0), (6, 40, 6, 20, 0), (9, 5, 6, 100, 0), (8, 2, 3, 256, 0), (8, 3, 2, 260, 0), (5, 4, 7, 26, 0), (6, 3, 8, 63, 0), (4, 6, 17, 65, 0),
    # fewer pairs than slices, whole chunks of 256 pairs and one more, few and many workgroups
    (1, 1, 6, 8, 0), (1, 256, 6, 8, 0), (1, 257, 6, 8, 0), (16, 32, 6, 100, 0), (32, 9, 6, 100, 0), (16, 20, 3, 45, 0),
    # wide slices: one tile of 49 to 64 lanes, two of 49 and of 33 with a ragged second, four of 64; the same through many passes
    (32, 3, 3, 63, 0), (32, 2, 3, 64, 0), (32, 2, 3, 97, 0), (32, 2, 3, 256, 0), (32, 2, 3, 126, 0), (32, 2, 3, 196, 0), (32, 2, 3, 260, 0), (32, 1, 2, 1024, 0), (12, 9, 57, 57, 0),
    # gz at a boundary of 8 and of 4 bytes with rows of whole groups of four
    (5, 6, 7, 100, 2), (5, 6, 7, 100, 1), (32, 2, 3, 64, 2), (32, 2, 3, 64, 1), (6, 40, 9, 4, 3)]


def vector_width(Fo, offset):
    return 4 if Fo % 4 == 0 and offset % 4 == 0 else 2 if Fo % 2 == 0 and offset % 2 == 0 else 1


def test_sizes_reach_the_splits_they_are_meant_for(split):
    seen = {}
    for nl, B, Fi, Fo, offset in SIZES:
        vec = vector_width(Fo, offset)
        lanes, slices = split(nl, B, Fi, Fo // vec)
        seen.setdefault(vec, []).append((lanes, slices, -(-(Fo // vec) // lanes), (Fo // vec) % lanes, (2 * nl - 1) * B))
    for vec in (1, 2, 4):
        lanes = {s[0] for s in seen[vec]}
        assert any(v == 4 for v in lanes) or vec == 2
        assert any(9 <= v <= 16 for v in lanes) and any(v > 48 for v in lanes), (vec, lanes)
        assert any(s[2] > 1 and s[3] for s in seen[vec]) or vec == 2                            # a ragged last tile
    every = [s for v in seen.values() for s in v]
    assert {4, 64} <= {s[0] for s in every} and any(17 <= s[0] <= 32 for s in every) and any(33 <= s[0] <= 48 for s in every)
    assert {1, 4, 51, 64} <= {s[1] for s in every}                                              # slices
    assert any(s[4] < 256 for s in every) and any(s[4] == 256 for s in every) and any(s[4] == 257 for s in every) and any(s[4] > 512 for s in every)


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo,offset", SIZES)
def test_kernel_gradient(hip, nl, B, Fi, Fo, offset):
    from s2cnn_amd.s2_real import s2_mm_real
    print(f"s2 kernel gradient nl={nl} B={B} Fi={Fi} Fo={Fo} offset={offset}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(nl)
    x = torch.randn(nl * nl, B, Fi, device="cuda", generator=g)
    y = torch.randn(nl * nl, Fi, Fo, device="cuda", generator=g).requires_grad_()
    z = s2_mm_real(x, y)
    gz = torch.randn(z.numel() + offset, device="cuda", generator=g)[offset:].view(z.shape)
    assert gz.is_contiguous() and gz.data_ptr() % 16 == 4 * offset
    (gy,) = torch.autograd.grad(z, y, gz)
    for l in range(nl):
        L, first = 2 * l + 1, l * (4 * l * l - 1) // 3
        want = torch.einsum("rsij,rik->skj", gz[first:first + L * L].view(L, L, B, Fo).double(), x[l * l:l * l + L].double())
        got = gy[l * l:l * l + L].double()
        # sums of L B products, at most one rounding of 2^-24 each on partial sums that grow with the root of their number
        assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -24 * (1 + (L * B) ** 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("nl,B,Fi,Fo", [(5, 7, 9, 8), (6, 3, 3, 63), (4, 80, 1, 6), (3, 1, 17, 4)])
def test_values_that_are_not_finite_stay_where_they_are(hip, nl, B, Fi, Fo):
    """Pairs beyond a slice's end and features beyond the last pass are loaded or multiplied, and must reach no result."""
    from s2cnn_amd.s2_real import s2_mm_real
    print(f"s2 kernel gradient, infinities, nl={nl} B={B} Fi={Fi} Fo={Fo}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(nl)
    x = torch.randn(nl * nl, B, Fi, device="cuda", generator=g)
    y = torch.randn(nl * nl, Fi, Fo, device="cuda", generator=g).requires_grad_()
    z = s2_mm_real(x, y)
    gz = torch.randn(z.shape, device="cuda", generator=g)
    for l in range(1, nl):                                       # one value in the first pair of a row, one in its last
        L, first = 2 * l + 1, l * (4 * l * l - 1) // 3
        gz[first, 0, 0] = float("inf")
        gz[first + L * (L - 1) + 1, B - 1, Fo - 1] = float("nan")
    (gy,) = torch.autograd.grad(z, y, gz)
    for l in range(nl):
        L, first = 2 * l + 1, l * (4 * l * l - 1) // 3
        want = (gz[first:first + L * L].view(L, L, B, 1, Fo).double() * x[l * l:l * l + L].view(L, 1, B, Fi, 1).double()).sum((0, 2))
        got = gy[l * l:l * l + L].double()
        finite = want.isfinite()
        assert torch.equal(got.isfinite(), finite) and torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isposinf(), want.isposinf())
        err = (got - want)[finite].norm() / want[finite].norm()
        assert err.item() <= 2.0 ** -24 * (1 + (L * B) ** 0.5)
