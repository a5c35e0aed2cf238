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
    assert 0 < a.matrix_frames <= 32 and b.matrix_frames == 0
    s = torch.cuda.Stream()
    img = torch.full((F,) + geom_c1.img_shape, float("nan"), dtype=torch.float32, device=cuda)
    with torch.cuda.stream(s):
        a(raw, planes, img, use_graph=True)   # a captured graph of the other path goes with it
    s.synchronize()
    a.variant = a.variant
    b.variant = a.variant
    assert a.matrix_frames == 0 and a.graph_count() == 0
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
    own, frames = a.variant, a.matrix_frames
    print(f"case: mixed C1, variant {own >> 8}, groups of {frames} frames on the matrix cores", flush=True)
    a.variant = own
    a.variant = own ^ 1                 # another FP32 variant, which this chain does not run
    assert a.matrix_frames == frames
    wide = next(v for v in range(device.bp_num_variants(True)) if device.bp_variant_shape(True, v)[1] == 32)
    a.variant = wide << 8
    assert a.matrix_frames == 0
    a.variant = own
    assert a.matrix_frames == frames
    a.close()
