"""FP16 backprojection of 64 slices on the matrix cores: the bits of the
16 x 16-tile variants of bp_linear_f16_kernel, and the mixed chain that uses it
for groups of 64 frames."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import FrameSet

pytestmark = pytest.mark.gpu


# partial tiles, angle counts around a chunk of 4 and a block of 64, detector
# counts that leave windows past either end, scales 0.6 .. 1.168 (rows of 2 and
# 4 angles per chunk), slices of a partial group and of one and both halves;
# values: normal, subnormal, and a few that are not finite
@pytest.mark.parametrize("N,P,D,rot,mask,S,kind", [
    (64, 20, 64, 0.0, 1, 64, "normal"), (97, 61, 101, 13.0, 0, 50, "normal"), (33, 1, 20, 45.0, 0, 1, "normal"),
    (250, 65, 292, -45.0, 1, 33, "normal"), (192, 130, 200, 0.0, 1, 64, "inf"), (96, 64, 96, -30.0, 1, 7, "tiny"),
    (512, 1000, 512, 0.0, 1, 64, "normal")])
def test_packed_equals_dot2(risa, geom_c0, cuda, N, P, D, rot, mask, S, kind):
    import torch
    from risa_amd import device

    lib = risa.load()
    run, size = lib.risa_bp_run_f16_packed, lib.risa_bp_f16_pack_bytes
    run.argtypes = [C.c_void_p, C.c_void_p, C.c_float, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
    run.restype = C.c_int
    size.argtypes, size.restype = [C.c_void_p], C.c_size_t
    print(f"case: packed FP16 BP N={N} P={P} D={D} rot={rot} S={S} {kind}", flush=True)
    g = geom_c0.replace(numberOfPixels=N, numberOfParallelProjections=P, numberOfParallelDetectors=D,
                        rotationOffset=rot, fusedMasking=mask, maskingValue=-3.0)
    bp = device.Backprojection(g)
    variants = [v for v in range(64) if _shape(device, v) and _shape(device, v)[:2] == (16, 16)]
    x = np.random.default_rng(N + D).standard_normal(((S + 3) // 4, P, D, 4))
    x = (x * (1e-6 if kind == "tiny" else 1.0)).astype(np.float16)
    if kind == "inf":
        x[3, 5, 77, 2], x[7, 9, 11, 1] = np.nan, np.inf
    if S % 4:
        x[-1, :, :, S % 4:] = 0
    x4 = torch.from_numpy(x.view(np.int16)).to(cuda)
    checked = 0
    for v in variants:
        bp.variant = v << 8
        if size(bp.h) == 0:   # groups of threads share the angles: another order of the sums
            continue
        want = torch.full((S, N, N), 7.0, dtype=torch.float32, device=cuda)
        bp.f16x4(x4, 4.0, S, want)
        img = torch.full((S + 1, N, N), 7.0, dtype=torch.float32, device=cuda)
        packed = torch.full((size(bp.h),), 0x7f, dtype=torch.uint8, device=cuda)   # halves that are NaN
        rc = run(bp.h, x4.data_ptr(), 4.0, S, packed.data_ptr(), img.data_ptr(), torch.cuda.current_stream().cuda_stream)
        assert rc == 0, lib.risa_last_error()
        torch.cuda.synchronize()
        assert bool((img[S] == 7.0).all())
        assert torch.equal(torch.isnan(img[:S]), torch.isnan(want)), f"variant {v}"
        assert torch.equal(torch.nan_to_num(img[:S], nan=5.0), torch.nan_to_num(want, nan=5.0)), f"variant {v}"
        checked += 1
    assert checked >= 1
    bp.close()


def _shape(device, v):
    try:
        return tuple(device.bp_variant_shape(True, v))
    except Exception:
        return None


def test_chain_mixed_large_groups(risa, geom_c1, cuda):
    """132 frames in groups of up to 64: every frame has the bits of a small
    chain with the same variants, eager and replayed as a graph with eager work
    between."""
    import torch
    from risa_amd import device

    fs = FrameSet(geom_c1, 1, 4, R=4)
    F = 132
    idx = np.arange(F) % 4
    raw = torch.from_numpy(fs.raw[idx]).to(cuda)
    planes = fs.planes[idx]
    a = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_MIXED, max_frames=F)
    b = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_MIXED, max_frames=4)
    b.variant = a.variant
    img = torch.full((F,) + geom_c1.img_shape, float("nan"), dtype=torch.float32, device=cuda)
    print(f"case: chain mixed C1, {F} frames, FP16 variant {a.variant >> 8}", flush=True)
    a(raw, planes, img)
    four = torch.empty((4,) + geom_c1.img_shape, dtype=torch.float32, device=cuda)
    for f in (0, 32, 60, 64, 124, 128):
        b(raw[f:f + 4], planes[f:f + 4], four)
        torch.cuda.synchronize()
        assert torch.equal(img[f:f + 4], four), f"frames {f} .. {f + 3}"
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
