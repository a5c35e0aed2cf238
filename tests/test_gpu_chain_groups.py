"""Chains that backproject groups of many frames on the matrix cores: which
frames take that path, and what pins or keeps it."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import FrameSet

pytestmark = pytest.mark.gpu


def _frames(g, cuda, F):
    import torch

    fs = FrameSet(g, 1, 4, R=4)
    idx = np.arange(F) % 4
    return fs, torch.from_numpy(fs.raw[idx]).to(cuda), fs.planes[idx]


def test_set_variant_pins_every_frame(risa, geom_c1, cuda):
    """A plain chain of 70 frames runs the matrix-core kernel until its own
    variant is set; then every frame of every call has the bits of a one-frame
    chain with that variant, eager and replayed."""
    import torch
    from risa_amd import device

    F = 70
    fs, raw, planes = _frames(geom_c1, cuda, F)
    a = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_PLAIN, max_frames=F)
    b = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_PLAIN, max_frames=1)
    assert a.on_matrix_cores(F) and not b.on_matrix_cores(1)
    s = torch.cuda.Stream()
    img = torch.full((F,) + geom_c1.img_shape, float("nan"), dtype=torch.float32, device=cuda)
    with torch.cuda.stream(s):
        a(raw, planes, img, use_graph=True)   # a captured graph of the other path goes with it
    s.synchronize()
    a.variant = a.variant
    b.variant = a.variant
    assert not a.on_matrix_cores(F) and a.graph_count() == 0
    print(f"case: plain C1, {F} frames, variant {a.variant & 0xff} set", flush=True)
    one = torch.empty((1,) + geom_c1.img_shape, dtype=torch.float32, device=cuda)
    for graph in (False, True):
        img.fill_(float("nan"))
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            a(raw, planes, img, use_graph=graph)
        s.synchronize()
        for f in (0, 31, 32, 63, 64, 69):
            b(raw[f:f + 1], planes[f:f + 1], one)
            torch.cuda.synchronize()
            assert torch.equal(one[0], img[f]), f"frame {f}"
    a.close()
    b.close()


def test_mixed_variants_keep_the_matrix_path(risa, geom_c1, cuda):
    """The mixed chain's matrix-core kernel has the bits of the 16 x 16 variants:
    it runs for those, and neither for another one nor only until one is set."""
    from risa_amd import device

    fs = FrameSet(geom_c1, 1, 2, R=2)
    a = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_MIXED, max_frames=128)
    own, frames = a.variant, a.on_matrix_cores(64)
    print(f"case: mixed C1, variant {own >> 8}, groups of 64 frames on the matrix cores: {frames}", flush=True)
    a.variant = own
    a.variant = own ^ 1                 # another FP32 variant, which this chain does not run
    assert a.on_matrix_cores(64) == frames
    wide = next(v for v in range(device.bp_num_variants(True)) if device.bp_variant_shape(True, v)[1] == 32)
    a.variant = wide << 8
    assert not a.on_matrix_cores(64)
    a.variant = own
    assert a.on_matrix_cores(64) == frames
    a.close()


def test_a_frames_place_does_not_matter(risa, geom_c1, cuda):
    """The same raw frame at every place of plain calls of several lengths: one
    image, bit for bit, within a call and for all calls of one way; the two
    ways within rounding of each other (5e-6, as the kernels)."""
    import torch
    from risa_amd import device

    F = 97
    fs, raw, _ = _frames(geom_c1, cuda, F)
    raw[:] = raw[0].clone()
    a = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_PLAIN, max_frames=F)
    assert a.on_matrix_cores(64)
    first = {}
    for n in (1, 2, 17, 32, 33, 64, 65, 70, 97):
        way = a.on_matrix_cores(n)
        print(f"case: plain C1, {n} equal frames, matrix cores: {way}", flush=True)
        img = torch.full((n,) + geom_c1.img_shape, float("nan"), dtype=torch.float32, device=cuda)
        a(raw[:n], np.zeros(n, np.int32), img)
        torch.cuda.synchronize()
        assert bool((img == img[0]).all())
        if way in first:
            assert torch.equal(img[0], first[way])
        first[way] = img[0]
    if len(first) == 2:
        assert float((first[True] - first[False]).norm() / first[False].norm()) < 5e-6
    a.close()


@pytest.mark.parametrize("N,P,D,S", [(64, 70, 61, 16), (48, 5, 50, 1), (130, 64, 100, 9)])
def test_few_slices_have_the_same_bits(risa, geom_c0, cuda, N, P, D, S):
    """Launches of up to 16 slices read half of each packed row: the bits of the
    same slices in a launch of 32."""
    import ctypes as C

    import torch
    from risa_amd import device

    lib = risa.load()
    run, size = lib.risa_bp_run_split, lib.risa_bp_split_bytes
    run.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_float, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
    run.restype, size.argtypes, size.restype = C.c_int, [C.c_void_p], C.c_size_t
    bp = device.Backprojection(geom_c0.replace(numberOfPixels=N, numberOfParallelProjections=P,
                                               numberOfParallelDetectors=D))
    x = torch.from_numpy(np.random.default_rng(N).standard_normal((32, P, D)).astype(np.float32)).to(cuda)
    packed = torch.full((size(bp.h),), 0x7f, dtype=torch.uint8, device=cuda)
    for shape in range(3):
        out = []
        for n in (32, S):
            out.append(torch.full((n + 1, N, N), 7.0, dtype=torch.float32, device=cuda))
            rc = run(bp.h, shape, x.data_ptr(), 1024.0, n, packed.data_ptr(), out[-1].data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
            assert rc == 0, lib.risa_last_error()
        torch.cuda.synchronize()
        assert torch.equal(out[0][:S], out[1][:S])
        assert bool((out[1][S] == 7.0).all() and (out[0][32] == 7.0).all())
    bp.close()


def test_packed_kernel_is_tried_whatever_shares_the_angles(risa, geom_c1, cuda):
    """The 64-slice kernel is timed for every 16 x 16 tile; where it is taken, a
    variant with shared angles gives way to one whose bits it has, and a variant
    of another tile stays and is not replaced."""
    import ctypes as C

    from risa_amd import device

    lib = risa.load()
    tune, size = lib.risa_bp_tune_f16_packed, lib.risa_bp_f16_pack_bytes
    tune.argtypes, tune.restype = [C.c_void_p, C.c_void_p, C.c_int, C.POINTER(C.c_int)], C.c_int
    size.argtypes, size.restype = [C.c_void_p], C.c_size_t
    bp = device.Backprojection(geom_c1)
    for v in range(device.bp_num_variants(True)):
        square = device.bp_variant_shape(True, v)[:2] == (16, 16)
        shared = lib.risa_bp_variant_groups(1, v) > 1
        bp.variant = v << 8
        n = C.c_int()
        assert tune(bp.h, None, 32, C.byref(n)) == 0, lib.risa_last_error()
        now = bp.variant >> 8
        print(f"case: FP16 variant {v} (16 x 16: {square}, shared angles: {shared}): packed from {n.value}, then {now}",
              flush=True)
        assert (n.value <= 64) == square   # 512^2 x 1000 angles: 11 us a slice, 14 and more with any variant
        if square:
            assert size(bp.h) > 0 and device.bp_variant_shape(True, now)[:2] == (16, 16)
        assert now == v or (square and shared)
    bp.close()


def test_extreme_counts_stay_in_range(risa, orc, geom_c0, cuda):
    """A plain call on the matrix cores with counts of 0 and 65535 side by side,
    dead detectors (reference at or below the dark current) and blank frames:
    finite, and near the float64 oracle.  Tolerance 1e-4: the FP32 angles (rounded
    by 2^-23) move a ray by up to 3e-5 of a sample at 256 pixels from the centre,
    neighbouring samples differ by up to twice their size."""
    import torch
    from conftest import rel_rmse
    from risa_amd import device

    g = geom_c0.replace(numberOfPixels=512, numberOfParallelDetectors=512, numberOfParallelProjections=300)
    Pf, Df = g.fan_shape
    rng = np.random.default_rng(3)
    ref = np.full((1, Pf, Df), 60000.0, np.float32)
    dark = np.full((1, Df), 300.0, np.float32)
    ref[0, :, 50:53], ref[0, :, 200] = 300.0, 100.0
    ref[0, 7, :] = 300.5
    F = 64
    raw = np.empty((F, Pf, Df), np.uint16)
    p, d = np.mgrid[0:Pf, 0:Df]
    for f in range(F):
        raw[f] = ((p + d + f) % 2 * 65535, rng.integers(0, 2, (Pf, Df)) * 65535, np.zeros((Pf, Df)),
                  np.full((Pf, Df), 65535))[f % 4]
    chain = device.Chain(g, ref, dark, mode=risa.CHAIN_PLAIN, max_frames=F)
    assert chain.on_matrix_cores(F)
    img = torch.full((F,) + g.img_shape, float("nan"), dtype=torch.float32, device=cuda)
    chain(torch.from_numpy(raw).to(cuda), np.zeros(F, np.int32), img)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(img).all())
    want = orc.Chain(g, ref, dark)
    for f in range(4):
        err = rel_rmse(img[f].cpu().numpy(), want.f64(raw[f], 0))
        print(f"case: extreme counts, frame {f}: rel RMSE against the oracle {err:.2e}", flush=True)
        assert err < 1e-4
    chain.close()


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_references_without_a_bound_keep_the_fp32_kernel(risa, geom_c1, cuda, bad):
    from risa_amd import device

    fs = FrameSet(geom_c1, 1, 1, R=2)
    ref = fs.avg_ref.copy()
    ref[1, 5, 17] = bad
    chain = device.Chain(geom_c1, ref, fs.avg_dark, mode=risa.CHAIN_PLAIN, max_frames=64)
    assert not chain.on_matrix_cores(64)
    chain.close()


def test_mixed_tail_on_the_matrix_cores(risa, geom_c1, cuda):
    """Groups of 64 and 61 frames, the last x4 group partly empty: the bits of a
    small chain with the same variants."""
    import torch
    from risa_amd import device

    F = 125
    fs, raw, planes = _frames(geom_c1, cuda, F)
    a = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_MIXED, max_frames=128)
    b = device.Chain(geom_c1, fs.avg_ref, fs.avg_dark, mode=risa.CHAIN_MIXED, max_frames=4)
    b.variant = a.variant
    square = device.bp_variant_shape(True, a.variant >> 8)[:2] == (16, 16)
    assert a.on_matrix_cores(61) == a.on_matrix_cores(64) == square   # from 49 frames on or fewer
    img = torch.full((F,) + geom_c1.img_shape, float("nan"), dtype=torch.float32, device=cuda)
    a(raw, planes, img)
    part = torch.empty((4,) + geom_c1.img_shape, dtype=torch.float32, device=cuda)
    for f in (0, 60, 64, 120):
        b(raw[f:f + 4], planes[f:f + 4], part)
        torch.cuda.synchronize()
        assert torch.equal(img[f:f + 4], part), f"frames {f} .. {f + 3}"
    b(raw[124:], planes[124:], part[:1])
    torch.cuda.synchronize()
    assert torch.equal(img[124], part[0])
    a.close()
    b.close()
