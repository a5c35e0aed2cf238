"""The FP32 backprojector on the matrix cores (bp_split_kernel, FP16 hi + lo
operands) against bp_linear_kernel, and the plain chain that uses it for
groups of 32 frames.

Tolerance: both kernels form t relative to an integer tile origin, at most one
apart, in float with |t| < 64, so their fractions differ by at most 2^-18 =
3.8e-6 a sample pair; with zero-mean samples of equal size the images differ by
less than that relative to their RMS, and the 22-bit operands add 2^-21 at
most.  5e-6 relative RMSE."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import FrameSet, rel_rmse

pytestmark = pytest.mark.gpu

TOL = 5e-6


def _split(lib):
    run, size = lib.risa_bp_run_split, lib.risa_bp_split_bytes
    run.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_float, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
    run.restype = C.c_int
    size.argtypes, size.restype = [C.c_void_p], C.c_size_t
    return run, size


# odd and even detector counts, images that are no multiple of a tile or of 4,
# angle counts that leave a partial group of 4, a partial chunk, one block of
# 64 records or several, scales 0.6 .. 1.168, every number of slices' edges
@pytest.mark.parametrize("N,P,D,rot,mask,S", [(512, 1000, 512, 0.0, 1, 32), (70, 97, 61, 13.0, 0, 5),
                                              (128, 36, 149, -30.0, 1, 31), (33, 7, 20, 45.0, 0, 1),
                                              (250, 65, 292, -45.0, 1, 17), (96, 130, 96, 0.0, 1, 16),
                                              (41, 1, 40, 5.0, 0, 2)])
def test_split_matches_linear(risa, geom_c0, cuda, N, P, D, rot, mask, S):
    import torch
    from risa_amd import device

    run, size = _split(risa.load())
    g = geom_c0.replace(numberOfPixels=N, numberOfParallelProjections=P, numberOfParallelDetectors=D,
                        rotationOffset=rot, fusedMasking=mask, maskingValue=-3.0)
    bp = device.Backprojection(g)
    x = torch.from_numpy(np.random.default_rng(N + D).standard_normal((S, P, D)).astype(np.float32)).to(cuda)
    want = torch.empty((S, N, N), dtype=torch.float32, device=cuda)
    bp.batch(x, S, want)
    packed = torch.full((size(bp.h),), 0x7f, dtype=torch.uint8, device=cuda)   # halves that are NaN
    for shape in range(3):
        print(f"case: split N={N} P={P} D={D} rot={rot} S={S} shape {shape}", flush=True)
        img = torch.full((S + 1, N, N), 7.0, dtype=torch.float32, device=cuda)
        rc = run(bp.h, shape, x.data_ptr(), 4096.0, S, packed.data_ptr(), img.data_ptr(),
                 torch.cuda.current_stream().cuda_stream)
        assert rc == 0, risa.load().risa_last_error()
        torch.cuda.synchronize()
        assert bool((img[S] == 7.0).all())
        err = max(rel_rmse(img[i].cpu().numpy(), want[i].cpu().numpy()) for i in range(S))
        print(f"  worst rel RMSE against the linear kernel {err:.2e}", flush=True)
        assert err < TOL
        if mask:
            assert torch.equal(img[:S] == -3.0, want == -3.0)
    bp.close()


def test_split_refuses_wide_scale(risa, geom_c0, cuda):
    from risa_amd import device

    _, size = _split(risa.load())
    for D, fits in ((149, True), (151, False)):   # scale 1.164 and 1.18 on 128 pixels
        bp = device.Backprojection(geom_c0.replace(numberOfPixels=128, numberOfParallelDetectors=D))
        assert (size(bp.h) > 0) == fits
        bp.close()


def test_chain_plain_large_groups(risa, geom_c1, cuda):
    """70 frames in groups of 32, 32 and 6: every frame within rounding of a
    one-frame chain's, eager and replayed as a graph with eager work between."""
    import torch
    from risa_amd import device

    fs = FrameSet(geom_c1, 1, 4, R=4)
    F = 70
    idx = np.arange(F) % 4
    raw = torch.from_numpy(fs.raw[idx]).to(cuda)
    planes = fs.planes[idx]
    a = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_PLAIN, max_frames=F)
    b = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_PLAIN, max_frames=1)
    img = torch.full((F,) + geom_c1.img_shape, float("nan"), dtype=torch.float32, device=cuda)
    print("case: chain plain C1, 70 frames", flush=True)
    a(raw, planes, img)
    one = torch.empty((1,) + geom_c1.img_shape, dtype=torch.float32, device=cuda)
    for f in (0, 1, 31, 32, 63, 64, 69):
        b(raw[f:f + 1], planes[f:f + 1], one)
        torch.cuda.synchronize()
        err = rel_rmse(img[f].cpu().numpy(), one[0].cpu().numpy())
        print(f"  frame {f}: rel RMSE against a single frame {err:.2e}", flush=True)
        assert err < TOL
    s = torch.cuda.Stream()
    again = torch.empty_like(img)
    for _ in range(3):
        img2 = torch.full_like(img, float("nan"))
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            a(raw, planes, img2, use_graph=True)
        s.synchronize()
        assert torch.equal(img2, img)
        a(raw, planes, again)
        torch.cuda.synchronize()
        assert torch.equal(again, img)
    a.close()
    b.close()


@pytest.mark.parametrize("N,P,S", [(33, 1, 1), (33, 3, 2), (40, 7, 3), (17, 13, 1), (64, 131, 5)])
def test_angle_groups(risa, geom_c0, cuda, N, P, S):
    """Variants whose angles are shared by groups of threads, with fewer angles
    than groups and uneven shares, against the first variant: every variant sums
    the same terms.  Bound 1e-5 of the image's norm: coordinates below 64 round
    to 4e-6, the sample differences they multiply are about 1.4 of a sample."""
    import torch
    from risa_amd import device

    g = geom_c0.replace(numberOfPixels=N, numberOfParallelProjections=P, numberOfParallelDetectors=N + 5)
    bp = device.Backprojection(g)
    x = torch.from_numpy(np.random.default_rng(N + P).standard_normal((S, P, N + 5)).astype(np.float32)).to(cuda)
    ref = None
    for v in range(device.bp_num_variants()):
        print(f"case: angle groups N={N} P={P} S={S} variant {v}", flush=True)
        bp.variant = v
        img = torch.full((S, N, N), float("nan"), dtype=torch.float32, device=cuda)
        bp.batch(x, S, img)
        torch.cuda.synchronize()
        ref = img if ref is None else ref
        assert float((img - ref).norm() / ref.norm()) < 1e-5
    bp.close()
