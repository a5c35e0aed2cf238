"""Tap gradient: the short sums after the row transforms, at the edges of
their workgroups."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,P,S", [
    (11, 1, 1),       # one row, fewer taps and bins than a wave
    (61, 700, 1),     # several hundred partials, taps a fraction of a workgroup
    (127, 41, 26),    # M = 256: the last bin is the Nyquist bin
    (509, 90, 12),    # more taps and bins than one workgroup's threads
])
def test_padded_tap_gradient_tail(risa, orc, geom_c0, cuda, D, P, S):
    """Against the FP64 oracle.  Bound 1e-5 in the 2-norm: a single-precision
    transform of length M <= 1100 rounds each bin to about eps log2 M = 1.2e-6
    of the spectrum's RMS, and the products' errors add over rows as randomly
    as the products do; the sums after the transforms run in double."""
    import torch
    from risa_amd import device

    print(f"case: padded tap gradient D={D} P={P} S={S}", flush=True)
    g = geom_c0.replace(numberOfParallelDetectors=D, numberOfParallelProjections=P)
    rng = np.random.default_rng(D + P + S)
    x = rng.standard_normal((S, P, D)).astype(np.float32)
    gr = (rng.standard_normal((S, P, D)) + 0.5 * x).astype(np.float32)
    flt = device.Filter(g)
    dt = torch.full((D // 2 + 1,), float("nan"), dtype=torch.float32, device=cuda)
    flt.grad_taps(torch.from_numpy(x).to(cuda), torch.from_numpy(gr).to(cuda), S, dt)
    torch.cuda.synchronize()
    ref = orc.grad_taps_f64(x.astype(np.float64), gr.astype(np.float64))
    err = float(np.linalg.norm(dt.cpu().numpy() - ref) / np.linalg.norm(ref))
    print(f"  rel L2 vs FP64 oracle {err:.2e}", flush=True)
    assert err < 1e-5
    flt.grad_taps(torch.from_numpy(x).to(cuda), torch.from_numpy(gr).to(cuda), 0, dt)   # no rows: zero
    torch.cuda.synchronize()
    assert float(dt.abs().max()) == 0.0
    flt.close()
