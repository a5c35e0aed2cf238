"""Rebinning of many frames of one plane: the frames of a launch are shared out
to several workgroups where the sinogram has few blocks."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,P,F", [(256, 500, 2), (256, 500, 13), (255, 500, 64), (31, 17, 67)])
def test_rebin_shared_frames_equal_single(risa, geom_c0, cuda, D, P, F):
    """Every frame of a batch has the bits it has alone (one workgroup per
    block either way, the same operations per output)."""
    import torch
    from risa_amd import device

    print(f"case: rebin D={D} P={P} frames={F}", flush=True)
    g = geom_c0.replace(numberOfParallelDetectors=D, numberOfParallelProjections=P)
    tables = device.Fan2Para(g)
    fan = torch.from_numpy(np.random.default_rng(F).random((F,) + tuple(g.fan_shape), dtype=np.float32)).to(cuda)
    got = torch.full((F, P, D), float("nan"), dtype=torch.float32, device=cuda)
    tables.batch(fan, [0] * F, got)
    one = torch.empty((P, D), dtype=torch.float32, device=cuda)
    for f in range(F):
        tables(fan[f], 0, one)
        torch.cuda.synchronize()
        assert torch.equal(one, got[f]), f"frame {f}"
    tables.close()
