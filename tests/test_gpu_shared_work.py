"""Work shared inside a launch: a plane's frames by several workgroups of the
rebinning, a pixel's angles by several groups of threads of the FP16
backprojector."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,P,planes", [(64, 40, "0111111101111"), (63, 40, "10" * 20 + "1" * 9), (63, 17, "1"),
                                        (128, 90, "0" * 33 + "1" * 40)])
def test_rebin_frames_of_two_planes(risa, geom_c1, cuda, D, P, planes):
    """Few blocks, so that both planes' frames (uneven numbers, in any order, odd
    D's extra column too) go to several workgroups: every frame has the bits it
    has alone."""
    import torch
    from risa_amd import device

    g = geom_c1.replace(numberOfParallelDetectors=D, numberOfParallelProjections=P)
    plane = [int(c) for c in planes]
    F = len(plane)
    print(f"case: rebin D={D} P={P}, {plane.count(0)} + {plane.count(1)} frames", flush=True)
    tables = device.Fan2Para(g)
    fan = torch.from_numpy(np.random.default_rng(F).random((F,) + tuple(g.fan_shape), dtype=np.float32)).to(cuda)
    got = torch.full((F + 1, P, D), 7.0, dtype=torch.float32, device=cuda)
    tables.batch(fan, plane, got[:F])
    one = torch.empty((P, D), dtype=torch.float32, device=cuda)
    for f in range(F):
        tables(fan[f], plane[f], one)
        torch.cuda.synchronize()
        assert torch.equal(one, got[f]), f"frame {f}"
    assert bool((got[F] == 7.0).all())
    tables.close()


@pytest.mark.parametrize("N,P,S", [(33, 1, 1), (33, 3, 6), (40, 7, 9), (9, 13, 4), (64, 131, 19)])
def test_fp16_angle_groups(risa, geom_c0, cuda, N, P, S):
    """FP16 variants with fewer angles than groups of threads, uneven shares,
    images below a tile and a partial group of slices, against the first variant.
    Bound 3e-4 of the image's norm: a weight f is rounded to FP16 (2^-12 at most)
    at a place that depends on the tile, times differences of about 1.4."""
    import torch
    from risa_amd import device

    g = geom_c0.replace(numberOfPixels=N, numberOfParallelProjections=P, numberOfParallelDetectors=N + 5)
    bp = device.Backprojection(g)
    x = np.random.default_rng(N + P).standard_normal(((S + 3) // 4, P, N + 5, 4)).astype(np.float16)
    if S % 4:
        x[-1, :, :, S % 4:] = 0
    x4 = torch.from_numpy(x.view(np.int16)).to(cuda)
    ref = None
    for v in range(device.bp_num_variants(True)):
        print(f"case: FP16 angle groups N={N} P={P} S={S} variant {v}", flush=True)
        bp.variant = v << 8
        img = torch.full((S + 1, N, N), 7.0, dtype=torch.float32, device=cuda)
        bp.f16x4(x4, 1.0, S, img)
        torch.cuda.synchronize()
        assert bool((img[S] == 7.0).all())
        ref = img if ref is None else ref
        assert float((img[:S] - ref[:S]).norm() / ref[:S].norm()) < 3e-4
    bp.close()
