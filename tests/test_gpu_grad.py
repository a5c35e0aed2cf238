"""The backward path and its transforms: rows of the filter and of the tap
gradient at each radix, row width and layout, the tap gradient's short sums at
the edges of their workgroups, and the adjoint projector's groups of images."""
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


@pytest.mark.parametrize("D", [1, 2, 3, 30, 16, 128, 250, 256, 500, 1024, 1280, 2048, 4000, 4096, 4608])
def test_filter_row_kernels(risa, orc, geom_c0, cuda, D):
    """The row transform at each radix, row width and LDS layout, and one
    length beyond LDS (4608), with an odd number of rows, against numpy in
    double.  Bound 2e-6 in the 2-norm: two transforms of at most 9 passes, each
    rounding to a few 6e-8 (twiddle, product, sums) of the RMS, added in
    quadrature: 3 x 6e-8 x sqrt(18) < 1e-6."""
    import torch
    from risa_amd import device

    print(f"case: filter rows D={D}", flush=True)
    P, S = 7, 3
    g = geom_c0.replace(numberOfParallelDetectors=D, numberOfParallelProjections=P)
    rng = np.random.default_rng(D)
    x = rng.standard_normal((S, P, D)).astype(np.float32)
    taps = (1.0 + rng.random(D // 2 + 1)).astype(np.float32)
    flt = device.Filter(g)
    flt.set_taps(taps)
    t = torch.from_numpy(x.copy()).to(cuda)
    flt(t, S)
    torch.cuda.synchronize()
    h = taps.astype(np.float64)
    ref = np.fft.irfft(np.fft.rfft(x.astype(np.float64)) * h, n=D) * D if D > 1 else x.astype(np.float64) * h[0]
    err = float(np.linalg.norm(t.cpu().numpy() - ref) / np.linalg.norm(ref))
    print(f"  rel L2 {err:.2e}", flush=True)
    assert err < 2e-6
    flt.close()


@pytest.mark.parametrize("D,rows", [(4, 3), (128, 5000), (256, 515), (500, 1100), (512, 1), (512, 5003), (1024, 700),
                                    (2048, 9)])
def test_tap_gradient_row_kernels(risa, orc, geom_c0, cuda, D, rows):
    """Lengths the transform takes unpadded: each row width, one to several rows
    per workgroup and pass, the register transform of 512; bound as above."""
    import torch
    from risa_amd import device

    print(f"case: tap gradient D={D} rows={rows}", flush=True)
    g = geom_c0.replace(numberOfParallelDetectors=D, numberOfParallelProjections=rows)
    rng = np.random.default_rng(D + rows)
    x = rng.standard_normal((1, rows, D)).astype(np.float32)
    gr = ((rng.standard_normal((1, rows, D)) + 0.5 * x) * 1e-5).astype(np.float32)
    flt = device.Filter(g)
    dt = torch.full((D // 2 + 1,), float("nan"), dtype=torch.float32, device=cuda)
    flt.grad_taps(torch.from_numpy(x).to(cuda), torch.from_numpy(gr).to(cuda), 1, dt)
    torch.cuda.synchronize()
    ref = orc.grad_taps_f64(x.astype(np.float64), gr.astype(np.float64))
    err = float(np.linalg.norm(dt.cpu().numpy() - ref) / np.linalg.norm(ref))
    print(f"  rel L2 vs FP64 oracle {err:.2e}", flush=True)
    assert err < 1e-5
    flt.close()


@pytest.mark.parametrize("N,P,mask", [(37, 5, True), (96, 18, False)])
def test_adjoint_image_groups(risa, geom_c0, cuda, N, P, mask):
    """The adjoint projector takes images in groups of four and a last two or
    one, and 16 per pass: every image's sinogram is the one it has alone, bit
    for bit (the same operations per image), also after a call that left other
    values, NaN among them, in the groups' buffers."""
    import torch
    from risa_amd import device

    g = geom_c0.replace(numberOfPixels=N, numberOfParallelProjections=P, numberOfParallelDetectors=N,
                        fusedMasking=int(mask))
    bp = device.Backprojection(g)
    x = torch.from_numpy(np.random.default_rng(N).standard_normal((19, N, N)).astype(np.float32)).to(cuda)
    alone = torch.empty((19, P, N), dtype=torch.float32, device=cuda)
    for i in range(19):
        bp.adjoint(x[i], alone[i])
    assert float(alone.abs().max()) > 0.0
    for S in (1, 2, 3, 4, 5, 6, 7, 16, 17, 19):
        print(f"case: adjoint groups N={N} slices={S}", flush=True)
        bad = torch.full((4, N, N), float("nan"), dtype=torch.float32, device=cuda)
        bp.adjoint_batch(bad, 4, torch.empty((4, P, N), dtype=torch.float32, device=cuda))
        got = torch.full((S, P, N), float("nan"), dtype=torch.float32, device=cuda)
        bp.adjoint_batch(x[:S].contiguous(), S, got)
        torch.cuda.synchronize()
        assert torch.equal(got, alone[:S])
    bp.close()
